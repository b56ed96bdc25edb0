// Host tables of the row solver (row_solve.hip): one workgroup solves one
// power flow, its lanes working on the grid's buses side by side.
//
// The Newton system is kept in 2 x 2 blocks, one per bus pair (a PV bus's
// second row and column are the identity's).  The buses are renumbered by
// their level in the elimination tree of the plan's pivot order (leaves 0; a
// bus's level is one above its highest child's), which is an elimination
// order of the same fill.  All buses of a level are eliminated together: the
// level's record list names every block (and right-hand side) that their
// rank-2 updates touch, once, with the terms that go into it, so each record
// is one thread's work, no two threads write the same place, and the sums
// come out in the same order every time.
#pragma once

#include <cstdint>
#include <vector>

#include "plan.hpp"

namespace g2g {

// record words: {target, first | count << 24, pivot block, term}, and in a list
// of its own {pivot block, term} of the second term
//   target  block index, or kRowRhs | bus for a right-hand side;
//           kRowInvert: the target is the diagonal block of a bus of the next
//           level, complete with these terms, and is replaced by its inverse
//   first   index of the record's third term
//   term    (L - D) | x << 8, x = U - D for a block, the pivot's bus for a right-hand side
constexpr int kRowInvert = 1 << 30;
constexpr int kRowRhs = 1 << 29;
constexpr int kRowMaxTerms = 127;   // terms of one record
constexpr int kRowMaxC = 63;        // off-diagonal blocks of one pivot
constexpr int kRowMaxLev = 127;     // elimination levels

struct RowPlan {
    bool ok = false;        // false: a bound of the record format does not hold
    int n = 0, nb = 0;      // buses; buses with unknowns, [0, nb) of the numbering (fixed buses follow)
    int n_blk = 0;          // 2 x 2 blocks
    int n_lev = 0;
    int n_slice = 0, n_fill = 0;
    std::vector<int> bus_of;     // [n] numbering -> bus
    std::vector<int> lev_ptr;    // [n_lev + 1] first bus of each level
    std::vector<int> rec_ptr;    // [n_lev + 1] first record of each level
    std::vector<int> lev_blk;    // [n_lev + 1] first block of each level's buses
    std::vector<int> rec;        // 4 words per record
    std::vector<int> rec2;       // 2 words per record: its second term
    std::vector<int> term;       // 2 words per further term: {pivot block, term}
    std::vector<int> back;       // 4 words per bus: {diagonal block, first | count << 24, two columns' buses (itself: none)}
    std::vector<int> back_col;   // buses of a pivot's third and further off-diagonal blocks
    // levels from which on no level has more records (buses) than a wavefront has lanes
    int solo_f = 0, solo_b = 0;
    std::vector<int> fill;       // blocks with no Ybus entry
    // mismatch: slices of 64 buses of like degree, entry q of a slice's bus at
    // [slice_ptr[s] + q][lane]
    std::vector<int> slice_ptr;  // [n_slice + 1]
    std::vector<int> slice_bus;  // 4 words per lane: {bus number (-1: none), diagonal block | PQ << 31, Ybus entry of the diagonal, bus}
    std::vector<int> ent;        // 4 words: {column's bus number, block << 2 | column PQ << 1 | row PQ (-1: none), Ybus entry, 0}
    std::vector<double> ent_y;   // 2 per entry
    std::vector<double> diag_y;  // 2 per lane
};

RowPlan build_row_plan(const NrPlan& P);

}  // namespace g2g
