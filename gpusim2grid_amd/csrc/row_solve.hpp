// Arguments of the row solver (row_solve.hip; tables: row_plan.hpp).
#pragma once

#include <hip/hip_runtime.h>

#include "device_common.hpp"

namespace g2g {

constexpr int kRowMaxEdits = 64;   // a row's Ybus edits kept in LDS
constexpr int kRowMaxThreads = 1024;
constexpr int kRowRedBytes = 8 * 8;  // the workgroup's maxima (two sets of two), the next slice, three clocks
// A row that ends unconverged with a residual above this (or not finite) is
// left as it came, for the tile kernels to finish: the iterates of a row that
// does not contract amplify rounding, so its last one is the solver's own, and
// callers keep getting the one they always got.  (Not in streamed rounds, where
// a row's V moves on with every launch.)
constexpr double kRowKeep = 1e-4;
// Such a row is given up early: from its third update here (or since its
// restart) on, when an update does not halve a residual above kRowKeep.  (By
// the oracle, from the flat start, 14 to 6,500 buses, injections scaled up to
// the last row that converges: every row that converges halves it or better
// from the third update on, nearly all others fail to by their fourth.)
constexpr int kRowLook = 3;
constexpr double kRowContract = 0.5;
constexpr int kRowGivenUp = 99;  // such a row's status inside the kernel

template <typename Real>
struct RowArgs {
    int n, nb, n_blk, n_lev, n_slice, n_fill, solo_f, solo_b;
    int blk_lds0;           // blocks [blk_lds0, n_blk) are kept in LDS ...
    int lev_lds;            // ... which are all of the levels' from this one on
    const int* bus_of;
    const int* lev_ptr;
    const int* rec_ptr;
    const int4* rec;
    const int2* rec2;
    const int2* term;
    const int4* back;
    const int* back_col;
    const int* fill;
    const int* slice_ptr;
    const int4* slice_bus;
    const int4* ent;
    const double2* ent_y;
    const double2* diag_y;
    double2* V;             // [T][n][64]
    const double2* S;
    RowEdits ed;            // ed.n_ed null: no edits
    const int* entry_row;   // [nY]
    int* status;
    int* iters;
    double* res;
    double* jmax;
    int row0, rows;         // rows [row0, rows)
    const int* list;        // nullable: the active rows; count at list_n
    const int* list_n;
    int iter0, skip_first;  // first iteration; 1: its statuses are already decided
    const int* clock;       // nullable: the first iteration is *clock + iter0 (streamed rounds)
    int max_upd;            // > 0: updates of one launch (a row not ended then stays active)
    int max_iter;
    double tol;
    int freeze;
    double growth, contraction;
    int look;               // kRowLook (streamed rounds, which hand no row back: never)
    double pivot_eps;
    int ir_steps;           // refinement rounds with the FP64 residual
    // learned starts (null without)
    const int* it0;
    int* budget;
    unsigned char* warm;
    const double2* V0;
    int v0_row, restart_max_iter;
    int* requeued;
    // per-workgroup scratch (blocks, V, refinement copies not kept in LDS)
    unsigned char* scratch;
    size_t scratch_stride;
    unsigned long long* updates;  // Newton updates summed over the rows
    int* last_iter;               // the largest iteration count
    int* left;                    // rows left as they came
    const int* stop;              // nullable: a launch before this left rows: leave all
    unsigned long long* clocks;   // [3] clocks of some rows' first step: mismatch, factorization, the rest (timed build)
};

constexpr size_t row_align(size_t v) { return (v + 31) / 32 * 32; }

// bytes of LDS without the blocks, and of scratch, per workgroup
template <typename Real>
size_t row_lds_bytes(int n, int nb, bool v_lds, bool edits)
{
    size_t s = row_align(kRowRedBytes) + row_align(static_cast<size_t>(nb) * 2 * sizeof(Real));
    if (v_lds) s += row_align(static_cast<size_t>(n) * sizeof(double2));
    if (edits)
        s += row_align(kRowMaxEdits * sizeof(double2)) + row_align(kRowMaxEdits * sizeof(int)) +
             row_align(static_cast<size_t>((n + 31) / 32) * 4);
    return s;
}
template <typename Real>
size_t row_scratch_bytes(int n, int nb, int blk_global, bool v_lds, bool refine)
{
    size_t s = static_cast<size_t>(blk_global) * 4 * sizeof(Real);
    if (!v_lds) s += row_align(static_cast<size_t>(n) * sizeof(double2));
    if (refine) s += static_cast<size_t>(nb) * 2 * sizeof(Real);
    return (s + 255) / 256 * 256;
}

template <typename Real, bool BL, bool VL, bool TIMED>
__global__ void k_row_solve(RowArgs<Real> a);
__global__ void k_collect_rows(const int* status, int rows, int* list, int* n);

}  // namespace g2g
