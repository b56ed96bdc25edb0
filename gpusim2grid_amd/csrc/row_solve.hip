// The row solver: one workgroup runs one power flow's whole Newton iteration.
//
// The tile kernels (kernels.hip) give a lane to a row and walk the grid's
// pivots one after the other, which fills the chip when there are thousands
// of rows and costs the whole walk however few there are.  Here the lanes of
// a workgroup share a row: the buses of one elimination level are independent
// (about half of a grid's buses are leaves, and 2,000 buses have 30 levels),
// so a factorization is one pass over the levels' update records with a
// barrier after each, a substitution one pass back, and the mismatch and the
// update are one pass over the buses.  The Newton loop, the status rule and
// the fallback of learned starts run inside, so a solve is one launch and no
// host round trip.
//
// What bounds it: the levels' dependent chain (record, terms' blocks, target,
// barrier): 2,000 buses mixed, one row, all in LDS, take 55 us an iteration,
// half of it the factorization's 30 levels, an eighth the substitution's.  The
// arithmetic is small (a 6,500-bus factorization is 17,785 updates of 2 x 2
// blocks).  6,500 buses FP64 (150 us an iteration) spend a third in the
// mismatch, whose V, tables and low blocks are in the L2.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "device_common.hpp"
#include "row_plan.hpp"
#include "row_solve.hpp"

namespace g2g {

namespace {

template <typename Real>
struct V4;
template <>
struct V4<float> {
    typedef float T __attribute__((ext_vector_type(4)));
};
template <>
struct V4<double> {
    typedef double T __attribute__((ext_vector_type(4)));
};

__device__ __forceinline__ double2 mul(double2 a, double2 b)
{
    return make_double2(fma(a.x, b.x, -a.y * b.y), fma(a.x, b.y, a.y * b.x));
}
// a conj(b)
__device__ __forceinline__ double2 mulc(double2 a, double2 b)
{
    return make_double2(fma(a.x, b.x, a.y * b.y), fma(a.y, b.x, -a.x * b.y));
}

// reciprocal: the hardware's, in FP64 with two Newton steps (x <- x + x (1 - d x)),
// which squares its relative error twice (an IEEE quotient is a chain twice as long)
__device__ __forceinline__ float inv_of(float d) { return __builtin_amdgcn_rcpf(d); }
__device__ __forceinline__ double inv_of(double d)
{
    double x = __builtin_amdgcn_rcp(d);
    x = fma(fma(-d, x, 1.0), x, x);
    return fma(fma(-d, x, 1.0), x, x);
}

// static-pivot clamp (own_lu/batched_lu.cu:45-53); NaN passes
template <typename Real>
__device__ __forceinline__ Real clamp_pivot(Real d, Real eps)
{
    return fabs(d) < eps ? (d < Real(0) ? -eps : eps) : d;
}

// The inverse of a diagonal block: its adjugate over its determinant, one
// reciprocal on the levels' dependent chain; with its two pivots taken in
// order (D00, then det / D00) where one of them is below the clamp.  Blocks
// are held column by column: {00, 10, 01, 11}.
template <typename Real>
__device__ __forceinline__ typename V4<Real>::T invert(typename V4<Real>::T D, Real eps)
{
    const Real det = fma(D[0], D[3], -D[2] * D[1]);
    const Real i = inv_of(det);
    typename V4<Real>::T R = {D[3] * i, -D[1] * i, -D[2] * i, D[0] * i};
    if (fabs(D[0]) < eps || fabs(det) < eps * fabs(D[0])) {
        const Real i1 = inv_of(clamp_pivot(D[0], eps));
        const Real l = D[1] * i1;
        const Real i2 = inv_of(clamp_pivot(fma(-l, D[2], D[3]), eps));
        const Real u = i1 * D[2] * i2;
        R = typename V4<Real>::T{fma(u, l, i1), -i2 * l, -u, i2};
    }
    return R;
}

__device__ __forceinline__ double nan_max(double m, double v)
{
    const double a = fabs(v);
    return (isnan(m) || isnan(a)) ? __builtin_nan("") : (a > m ? a : m);
}

constexpr int kGroup = 4;  // Ybus entries of a bus gathered together

}  // namespace

// the active rows' indices, in any order (each row's result is its own)
__global__ void k_collect_rows(const int* status, int rows, int* list, int* n)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < rows && status[r] == kActive) list[atomicAdd(n, 1)] = r;
}

// BL: every block in LDS; else the blocks below blk_lds0 (the lowest levels,
// where most blocks and the least dependence are) are in the workgroup's
// scratch.  VL: V in LDS, else in the scratch.  TIMED: with the phases' clocks.
template <typename Real, bool BL, bool VL, bool TIMED>
__global__ __launch_bounds__(kRowMaxThreads) void k_row_solve(RowArgs<Real> a)
{
    using B4 = typename V4<Real>::T;
    using R2 __attribute__((ext_vector_type(2))) = Real;
    const int tid = threadIdx.x, nt = blockDim.x;
    const int lane = tid & (kLanes - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kLanes), n_wave = nt / kLanes;
    extern __shared__ __align__(32) unsigned char g2g_row_smem[];
    unsigned char* at = g2g_row_smem;
    auto take = [&](size_t bytes) {
        unsigned char* p = at;
        at += row_align(bytes);
        return p;
    };
    auto* red = reinterpret_cast<unsigned long long*>(take(kRowRedBytes));
    int* slice_next = reinterpret_cast<int*>(red + 4);
    Real* b = reinterpret_cast<Real*>(take(static_cast<size_t>(a.nb) * 2 * sizeof(Real)));
    R2* b2 = reinterpret_cast<R2*>(b);
    const bool edits = a.ed.n_ed != nullptr;
    double2* ed_val = nullptr;
    int* ed_ent = nullptr;
    unsigned* ed_map = nullptr;
    if (edits) {
        ed_val = reinterpret_cast<double2*>(take(kRowMaxEdits * sizeof(double2)));
        ed_ent = reinterpret_cast<int*>(take(kRowMaxEdits * sizeof(int)));
        ed_map = reinterpret_cast<unsigned*>(take(static_cast<size_t>((a.n + 31) / 32) * 4));
    }
    unsigned char* sc = a.scratch + blockIdx.x * a.scratch_stride;
    double2* V;
    if constexpr (VL) {
        V = reinterpret_cast<double2*>(take(static_cast<size_t>(a.n) * sizeof(double2)));
    } else {
        V = reinterpret_cast<double2*>(sc);
        sc += row_align(static_cast<size_t>(a.n) * sizeof(double2));  // (B4 is 32 bytes in FP64)
    }
    B4* const ML = reinterpret_cast<B4*>(at);  // the LDS blocks
    B4* const MG = reinterpret_cast<B4*>(sc);
    const int lds0 = a.blk_lds0;
    // block q: known to be in LDS (levels from lev_lds on), or wherever it is
    auto blk = [&](auto in_lds, int q) -> B4* {
        if constexpr (BL) return ML + q;
        else if constexpr (decltype(in_lds)::value) return ML + (q - lds0);
        else return q >= lds0 ? ML + (q - lds0) : MG + q;
    };
    const std::false_type anywhere{};
    const std::true_type in_lds{};
    auto load = [&](int q) -> B4 { return *blk(anywhere, q); };
    auto store = [&](int q, B4 v) { *blk(anywhere, q) = v; };
    if constexpr (!BL) sc += static_cast<size_t>(lds0) * sizeof(B4);
    Real* xs = reinterpret_cast<Real*>(sc);  // refinement: the step so far
    // the level pointers, a lane each of two registers
    auto lane_of = [&](const int* p, int l) { return p[l <= a.n_lev ? l : a.n_lev]; };
    const int rp0 = lane_of(a.rec_ptr, lane), rp1 = lane_of(a.rec_ptr, kLanes + lane);
    const int lp0 = lane_of(a.lev_ptr, lane), lp1 = lane_of(a.lev_ptr, kLanes + lane);
    auto rec_ptr = [&](int l) {
        return l < kLanes ? __builtin_amdgcn_readlane(rp0, l) : __builtin_amdgcn_readlane(rp1, l - kLanes);
    };
    auto lev_ptr = [&](int l) {
        return l < kLanes ? __builtin_amdgcn_readlane(lp0, l) : __builtin_amdgcn_readlane(lp1, l - kLanes);
    };
    // Barriers that order the LDS only: loads of records for the next level
    // stay in flight across them (a full barrier waits for every load and
    // store of global memory, an L2 round trip a level).  Enough between
    // levels whose blocks are all in LDS.
    auto lds_sync = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    auto sync = [&](bool lds) {
        if (BL || lds) lds_sync();
        else __syncthreads();
    };
    // the same for a wavefront's own writes and reads
    auto wave_sync = [&](bool lds) {
        if (BL || lds) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup", "local");
        else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        __builtin_amdgcn_wave_barrier();
    };
    const int lev_lds = BL ? 0 : a.lev_lds;
    // a wavefront's next slice of buses: the first by its number, then
    // whichever is left (the first slices hold the buses of highest degree)
    auto next_slice = [&]() {
        int s = 0;
        if (lane == 0) s = atomicAdd(slice_next, 1);
        return __builtin_amdgcn_readfirstlane(s);
    };

    // where the time goes: the clocks of the phases of the workgroup's first
    // Newton step, in LDS; `ends` stops at this moment and `begins` starts.  A
    // build of its own: with it every power flow of 118 buses takes 1.5 to 3 us
    // longer, also where a flag switches the clocks off.
    unsigned long long* const clk = red + 5;
    auto lap = [&](bool now, int ends, int begins) {
        if constexpr (TIMED) {
            if (!now || tid != 0) return;
            const unsigned long long t = __builtin_readcyclecounter();
            if (ends >= 0) clk[ends] += t;
            if (begins >= 0) clk[begins] -= t;
        }
    };
    if (TIMED && tid < 3) clk[tid] = 0ull;
    const int todo = a.list ? *a.list_n : a.rows - a.row0;
    if (a.stop && *a.stop > 0) {
        if (blockIdx.x == 0 && tid == 0) atomicAdd(a.left, todo);
        return;
    }
    for (int i = blockIdx.x; i < todo; i += gridDim.x) {
        int row = a.row0 + i;
        if (a.list) {
            row = a.list[i];
        } else if (gridDim.x % 64 == 0 && i - static_cast<int>(blockIdx.x) + static_cast<int>(gridDim.x) <= todo) {
            // workgroup g runs on XCD g % 8: rows 8 r .. 8 r + 7, whose V and
            // Sbus share cache lines, go to one XCD's workgroups
            const int g = blockIdx.x, s = g / kXcds;
            row = a.row0 + i - g + ((s / 8) * kXcds + g % kXcds) * 8 + s % 8;
        }
        if (!a.list && a.status[row] != kActive) continue;
        const size_t tile = static_cast<size_t>(row) / kLanes;
        const int rl = row % kLanes;
        const size_t vbase = tile * a.n * kLanes + rl;
        int n_ed = 0;
        __syncthreads();  // the row before is done with the LDS
        for (int q = tid; q < a.n; q += nt) V[q] = a.V[vbase + static_cast<size_t>(a.bus_of[q]) * kLanes];
        if (edits) {
            n_ed = a.ed.n_ed[row];
            for (int q = tid; q < (a.n + 31) / 32; q += nt) ed_map[q] = 0u;
            __syncthreads();
            for (int q = tid; q < n_ed; q += nt) {
                const size_t e = (tile * a.ed.cap + q) * kLanes + rl;
                const int en = a.ed.ent[e];
                ed_ent[q] = en;
                ed_val[q] = a.ed.val[e];
                const int bus = a.entry_row[en];
                atomicOr(&ed_map[bus >> 5], 1u << (bus & 31));
            }
        }
        const int it0 = a.it0 ? a.it0[row] : 0;
        int budget = a.budget ? a.budget[row] : a.max_iter;
        bool wrow = a.warm && a.warm[row], restarted = false;
        double prev = a.res[row];
        double growth = a.growth;
        bool decide = !a.skip_first;
        int iter = a.clock ? *a.clock + a.iter0 : a.iter0, st = kActive, n_upd = 0;
        double jm = 0.0;
        int turn = 0, look = iter - it0 + a.look;  // look: the update from which on a row must contract
        if (tid == 0) {
            *slice_next = n_wave;
            red[0] = red[1] = 0ull;
        }
        __syncthreads();

        // a Ybus value less the row's edits of entry k
        auto edited = [&](int k, double2 y) {
            for (int t = 0; t < n_ed; ++t)
                if (ed_ent[t] == k) {
                    y.x -= ed_val[t].x;
                    y.y -= ed_val[t].y;
                }
            return y;
        };
        // One record: a block's (blocks) or a right-hand side's updates by a
        // level's pivots.  A right-hand side is run as a block whose two
        // columns are both the vector: the same loads, arithmetic and stores
        // (its two stores write one value to one place), so a wavefront of
        // mixed records has no divergent path, and all its LDS reads go out
        // together (under a condition each path's would be waited for where
        // the paths join).  A solve so, against a branch for each kind: 118 FP64
        // 4,096 rows 0.28 / 0.30 ms; 2,000 mixed 777 rows 0.80 / 0.90.
        auto update = [&](auto in, const int4 rec, const int2 rec2, Real eps, bool blocks) {
            const int tgt = rec.x & (kRowRhs - 1), cnt = rec.y >> 24, first = rec.y & 0xFFFFFF;
            const bool rhs = rec.x & kRowRhs;
            if (!rhs && !blocks) return;
            auto column = [&](int q) { return rhs ? b2 + q : reinterpret_cast<R2*>(blk(in, rhs ? 0 : q)); };
            const int second = rhs ? 0 : 1;
            R2* const p0 = column(tgt);
            R2* const p1 = p0 + second;
            R2 t0 = *p0, t1 = *p1;
            auto term = [&](int d, int w) {
                const R2* u = column(rhs ? w >> 8 : d + (w >> 8));
                const B4 L = *blk(in, d + (w & 0xFF)), D = *blk(in, d);
                const R2 u0 = u[0], u1 = u[second];
                const Real w00 = fma(D[0], u0[0], D[2] * u0[1]), w01 = fma(D[0], u1[0], D[2] * u1[1]);
                const Real w10 = fma(D[1], u0[0], D[3] * u0[1]), w11 = fma(D[1], u1[0], D[3] * u1[1]);
                t0[0] = fma(-L[0], w00, fma(-L[2], w10, t0[0]));
                t1[0] = fma(-L[0], w01, fma(-L[2], w11, t1[0]));
                t0[1] = fma(-L[1], w00, fma(-L[3], w10, t0[1]));
                t1[1] = fma(-L[1], w01, fma(-L[3], w11, t1[1]));
            };
            term(rec.z, rec.w);
            if (cnt > 1) {
                term(rec2.x, rec2.y);
                for (int e = 2; e < cnt; ++e) {
                    const int2 tm = a.term[first + e - 2];
                    term(tm.x, tm.y);
                }
            }
            if (rec.x & kRowInvert) {
                const B4 v = invert<Real>(B4{t0[0], t0[1], t1[0], t1[1]}, eps);
                t0 = R2{v[0], v[1]};
                t1 = R2{v[2], v[3]};
            }
            *p0 = t0;
            *p1 = t1;
        };
        // factorization and forward substitution (blocks), or the latter alone:
        // the wide levels by every thread with a barrier after each, the
        // narrow ones above (no more records than lanes) by one wavefront
        // with none.  A level's first records are loaded before the wait for
        // the level below it (always loaded, at a clamped index: a load under
        // a condition would be waited for where its paths join).
        auto eliminate = [&](Real eps, bool blocks) {
            const int last = a.n_lev - 1, solo = a.solo_f < last ? a.solo_f : last;
            if (last > 0) {
                const int n_rec = rec_ptr(a.n_lev);
                int4 rec;
                int2 rec2;
                auto fetch = [&](int q) {
                    const int at = q < n_rec ? q : n_rec - 1;
                    rec = a.rec[at];
                    rec2 = a.rec2[at];
                };
                int end = rec_ptr(1);
                fetch(tid);
                auto wide = [&](auto in, int l) {
                    for (int q = rec_ptr(l) + tid; q < end; q += nt) {
                        const int4 now = rec;
                        const int2 now2 = rec2;
                        fetch(q + nt < end ? q + nt : end + tid);
                        update(in, now, now2, eps, blocks);
                    }
                    if (rec_ptr(l) + tid >= end) fetch(end + tid);  // (no record of this level)
                    end = rec_ptr(l + 2 <= a.n_lev ? l + 2 : a.n_lev);
                };
                for (int l = 0; l < solo; ++l) {
                    if (BL || l >= lev_lds) wide(in_lds, l);
                    else wide(anywhere, l);
                    sync(l + 1 >= lev_lds);
                }
                if (wave == 0) {
                    for (int l = solo; l < last; ++l) {
                        const int4 now = rec;
                        const int2 now2 = rec2;
                        const bool mine = rec_ptr(l) + lane < end;
                        fetch(end + lane);
                        end = rec_ptr(l + 2 <= a.n_lev ? l + 2 : a.n_lev);
                        if (mine) {
                            if (BL || l >= lev_lds) update(in_lds, now, now2, eps, blocks);
                            else update(anywhere, now, now2, eps, blocks);
                        }
                        wave_sync(l + 1 >= lev_lds);
                    }
                }
            }
            sync(solo >= lev_lds);
        };
        // x over b, level by level from the top: the narrow levels by one
        // wavefront, the wide ones by every thread
        // (the first two columns' reads go out with the pivot's; a missing
        // column reads the pivot's own block, times zero)
        auto solve_bus = [&](auto in, int k, const int4 r) {
            const int c = r.y >> 24, first = r.y & 0xFFFFFF;
            R2 t = b2[k];
            const B4 D = *blk(in, r.x);
            const B4 U0 = *blk(in, c > 0 ? r.x + 2 : r.x), U1 = *blk(in, c > 1 ? r.x + 4 : r.x);
            R2 x0 = b2[r.z], x1 = b2[r.w];
            if (c < 1) x0 = R2{Real(0), Real(0)};
            if (c < 2) x1 = R2{Real(0), Real(0)};
            auto sub = [&](const B4& U, const R2& x) {
                t[0] = fma(-U[0], x[0], fma(-U[2], x[1], t[0]));
                t[1] = fma(-U[1], x[0], fma(-U[3], x[1], t[1]));
            };
            sub(U0, x0);
            sub(U1, x1);
            for (int q = 2; q < c; ++q) sub(*blk(in, r.x + 2 + 2 * q), b2[a.back_col[first + q - 2]]);
            R2 x;
            x[0] = fma(D[0], t[0], D[2] * t[1]);
            x[1] = fma(D[1], t[0], D[3] * t[1]);
            b2[k] = x;
        };
        auto substitute = [&]() {
            const int solo = a.solo_b;  // levels [solo, n_lev) by wavefront 0
            auto fetch = [&](int k) { return a.back[k < a.nb ? k : a.nb - 1]; };
            if (wave == 0 && solo < a.n_lev) {
                int end = a.nb, begin = lev_ptr(a.n_lev - 1);
                int4 r = fetch(begin + lane);
                for (int l = a.n_lev - 1; l >= solo; --l) {
                    const int4 now = r;
                    const int k = begin + lane;
                    const bool mine = k < end;
                    end = begin;
                    begin = lev_ptr(l > 0 ? l - 1 : 0);
                    r = fetch(begin + lane);
                    if (mine) {
                        if (BL || l >= lev_lds) solve_bus(in_lds, k, now);
                        else solve_bus(anywhere, k, now);
                    }
                    wave_sync(true);
                }
            }
            int4 r = fetch(solo > 0 ? lev_ptr(solo - 1) + tid : 0);
            lds_sync();
            for (int l = solo - 1; l >= 0; --l) {
                const int end = lev_ptr(l + 1), below = lev_ptr(l > 0 ? l - 1 : 0) + tid;
                int k = lev_ptr(l) + tid;
                if (k < end) {
                    auto wide = [&](auto in) {
                        for (; k < end; k += nt) {
                            const int4 now = r;
                            r = fetch(k + nt < end ? k + nt : below);
                            solve_bus(in, k, now);
                        }
                    };
                    if (BL || l >= lev_lds) wide(in_lds);
                    else wide(anywhere);
                } else {
                    r = fetch(below);
                }
                lds_sync();
            }
        };

        for (;;) {
            const bool timed = TIMED && i == static_cast<int>(blockIdx.x) && n_upd == 0 && !restarted;
            lap(timed, -1, 0);
            // F and J at V
            double rmax = 0.0, jmax = 0.0;
            for (int q = tid; q < a.n_fill; q += nt) store(a.fill[q], B4{Real(0), Real(0), Real(0), Real(0)});
            for (int s = wave; s < a.n_slice; s = next_slice()) {
                const int4 sb = a.slice_bus[s * kLanes + lane];
                const int e0 = a.slice_ptr[s], e1 = a.slice_ptr[s + 1];
                const int k = sb.x < 0 ? 0 : sb.x;
                const double2 vi = V[k];
                const double2 S = a.S[vbase + static_cast<size_t>(sb.w) * kLanes];
                double2 yd = a.diag_y[s * kLanes + lane];
                const bool ed = n_ed > 0 && (ed_map[sb.w >> 5] >> (sb.w & 31) & 1u);
                if (ed) yd = edited(sb.z, yd);
                const double2 t0 = mul(yd, vi);
                double2 I = t0;
                // kGroup entries' loads are issued before the first is used
                for (int eb = e0; eb < e1; eb += kGroup) {
                    int4 en[kGroup];
                    double2 y[kGroup], vj[kGroup];
#pragma unroll
                    for (int g = 0; g < kGroup; ++g) {
                        const int e = (eb + g < e1 ? eb + g : e1 - 1) * kLanes + lane;
                        en[g] = a.ent[e];
                        y[g] = a.ent_y[e];
                    }
#pragma unroll
                    for (int g = 0; g < kGroup; ++g) vj[g] = V[en[g].x];
#pragma unroll
                    for (int g = 0; g < kGroup; ++g) {
                        if (eb + g >= e1) break;
                        if (ed) y[g] = edited(en[g].z, y[g]);
                        const double2 t = mul(y[g], vj[g]);
                        I.x += t.x;
                        I.y += t.y;
                        if (en[g].y < 0) continue;
                        // dS_i / d theta_j = (w.y, -w.x), dS_i / dVm_j x |V_j| = (w.x, w.y), w = V_i conj(Y_ij V_j)
                        const double2 w = mulc(vi, t);
                        const Real wx = static_cast<Real>(w.x), wy = static_cast<Real>(w.y);
                        const bool rq = en[g].y & 1, cq = en[g].y & 2;
                        store(en[g].y >> 2, B4{wy, rq ? -wx : Real(0), cq ? wx : Real(0), rq && cq ? wy : Real(0)});
                        jmax = fmax(jmax, fmax(fabs(w.x), fabs(w.y)));
                    }
                }
                if (sb.x >= 0) {
                    const bool q = sb.y < 0;
                    const double2 sc2 = mulc(vi, I);
                    const double fp = -(sc2.x - S.x), fq = q ? -(sc2.y - S.y) : 0.0;
                    rmax = nan_max(nan_max(rmax, fp), fq);
                    b2[k] = R2{static_cast<Real>(fp), static_cast<Real>(fq)};
                    const double2 z = mulc(vi, make_double2(I.x - t0.x, I.y - t0.y));
                    const double2 u = mulc(vi, make_double2(I.x + t0.x, I.y + t0.y));
                    jmax = fmax(jmax, fmax(fmax(fabs(z.x), fabs(z.y)), fmax(fabs(u.x), fabs(u.y))));
                    store(sb.y & 0x7FFFFFFF, q ? B4{static_cast<Real>(-z.y), static_cast<Real>(z.x),
                                                    static_cast<Real>(u.x), static_cast<Real>(u.y)}
                                               : B4{static_cast<Real>(-z.y), Real(0), Real(0), Real(1)});
                }
            }
            // the workgroup's maxima: of magnitudes, whose bit patterns order as
            // unsigned numbers with NaN above all (a NaN anywhere makes r NaN).
            // Two sets of cells take turns: one is cleared while the other is read.
            auto bits = [](double v) { return static_cast<unsigned long long>(__double_as_longlong(v)); };
            for (int o = 32; o > 0; o >>= 1) {
                rmax = nan_max(rmax, __shfl_xor(rmax, o, 64));
                jmax = fmax(jmax, __shfl_xor(jmax, o, 64));
            }
            unsigned long long* const cell = red + turn;
            if (lane == 0) {
                atomicMax(cell, bits(rmax));
                atomicMax(cell + 1, bits(jmax));
            }
            __syncthreads();
            const double r = __longlong_as_double(static_cast<long long>(cell[0]));
            jm = __longlong_as_double(static_cast<long long>(cell[1]));
            turn ^= 2;
            if (tid == 0) {
                *slice_next = n_wave;
                red[turn] = red[turn + 1] = 0ull;
            }
            // the status rule (kernels.hip mis_status)
            const int it = iter - it0;
            if (decide) {
                const bool growth_on = growth > 0.0 && (!a.warm || wrow);
                if (!isfinite(r)) st = wrow ? kRejected : kDiverged;
                else if (a.freeze && r < a.tol) st = kConverged;
                else if (growth_on && it > 0 && r > growth * prev) st = kRejected;
                else if (wrow && growth > 0.0 && a.contraction > 0.0 && it >= 2 && r >= a.tol &&
                         r > a.contraction * prev * prev)
                    st = kRejected;
                else if (it >= budget) st = r < a.tol ? kConverged : (wrow ? kRejected : kMaxIter);
                // (not a row on a learned start, which has its own rejection rule)
                else if (it >= look && !wrow && r > kRowContract * prev && r >= kRowKeep) st = kRowGivenUp;
            }
            prev = r;
            if (st == kRejected && wrow) {
                // a learned start that failed: the fallback start, at this iteration
                wrow = false;
                budget = it + a.restart_max_iter;
                restarted = true;
                look = it + a.look;
                for (int q = tid; q < a.n; q += nt) {
                    const int bus = a.bus_of[q];
                    V[q] = a.v0_row ? a.V0[bus] : a.V0[vbase + static_cast<size_t>(bus) * kLanes];
                }
                st = kActive;
                growth = 0.0;
                decide = true;
                __syncthreads();
                continue;
            }
            lap(timed, 0, 1);
            if (st != kActive || it >= a.max_iter) break;
            growth = a.growth;
            decide = true;
            const Real eps = static_cast<Real>(a.pivot_eps) * static_cast<Real>(jm);
            for (int k = tid; k < lev_ptr(1); k += nt) {
                const int d = a.back[k].x;
                store(d, invert<Real>(load(d), eps));
            }
            sync(lev_lds == 0);
            eliminate(eps, true);
            lap(timed, 1, 2);
            substitute();
            for (int ir = 0; ir < a.ir_steps; ++ir) {
                // r = F(V) - J(V) dx in FP64, dV_j = V_j (dVm_j / |V_j| + j dtheta_j); then J d = r
                for (int q = tid; q < 2 * a.nb; q += nt) xs[q] = ir == 0 ? b[q] : xs[q] + b[q];
                __syncthreads();
                R2* x2 = reinterpret_cast<R2*>(xs);
                auto dv = [&](int k) {
                    if (k >= a.nb) return make_double2(0.0, 0.0);
                    const R2 x = x2[k];
                    return mul(V[k], make_double2(static_cast<double>(x[1]), static_cast<double>(x[0])));
                };
                for (int s = wave; s < a.n_slice; s = next_slice()) {
                    const int4 sb = a.slice_bus[s * kLanes + lane];
                    const int e0 = a.slice_ptr[s], e1 = a.slice_ptr[s + 1];
                    const int k = sb.x < 0 ? 0 : sb.x;
                    const double2 vi = V[k], dvi = dv(k);
                    const double2 S = a.S[vbase + static_cast<size_t>(sb.w) * kLanes];
                    double2 yd = a.diag_y[s * kLanes + lane];
                    const bool ed = n_ed > 0 && (ed_map[sb.w >> 5] >> (sb.w & 31) & 1u);
                    if (ed) yd = edited(sb.z, yd);
                    double2 I = mul(yd, vi), dI = mul(yd, dvi);
                    for (int e = e0; e < e1; ++e) {
                        const int4 en = a.ent[e * kLanes + lane];
                        double2 y = a.ent_y[e * kLanes + lane];
                        if (ed) y = edited(en.z, y);
                        const double2 t = mul(y, V[en.x]), u = mul(y, dv(en.x));
                        I.x += t.x;
                        I.y += t.y;
                        dI.x += u.x;
                        dI.y += u.y;
                    }
                    if (sb.x >= 0) {
                        const double2 sc2 = mulc(vi, I), p = mulc(dvi, I), u = mulc(vi, dI);
                        const double rp = -(sc2.x - S.x) - (p.x + u.x);
                        const double rq = sb.y < 0 ? -(sc2.y - S.y) - (p.y + u.y) : 0.0;
                        b2[k] = R2{static_cast<Real>(rp), static_cast<Real>(rq)};
                    }
                }
                __syncthreads();
                if (tid == 0) *slice_next = n_wave;
                eliminate(eps, false);
                substitute();
                if (ir + 1 == a.ir_steps) {
                    for (int q = tid; q < 2 * a.nb; q += nt) b[q] = xs[q] + b[q];
                    __syncthreads();
                }
            }
            for (int k = tid; k < a.nb; k += nt) {
                const R2 x = b2[k];
                const double m = 1.0 + static_cast<double>(x[1]);
                double sn, cs;
                sincos(static_cast<double>(x[0]), &sn, &cs);
                V[k] = mul(V[k], make_double2(m * cs, m * sn));
            }
            ++iter;
            ++n_upd;
            __syncthreads();
            lap(timed, 2, -1);
            if (a.max_upd > 0 && n_upd >= a.max_upd) break;  // st: still active
        }
        if (!a.clock && st != kConverged && !(prev < kRowKeep)) {
            if (tid == 0) atomicAdd(a.left, 1);
            continue;
        }
        for (int k = tid; k < a.nb; k += nt) a.V[vbase + static_cast<size_t>(a.bus_of[k]) * kLanes] = V[k];
        if (tid == 0) {
            a.res[row] = prev;
            a.jmax[row] = jm;
            if (st != kActive) {
                a.status[row] = st;
                a.iters[row] = iter - it0;
            }
            if (a.warm) {
                a.warm[row] = wrow ? 1 : 0;
                a.budget[row] = budget;
            }
            if (restarted) atomicAdd(a.requeued, 1);
            if (n_upd) atomicAdd(a.updates, static_cast<unsigned long long>(n_upd));
            atomicMax(a.last_iter, iter);
        }
    }
    if constexpr (TIMED) {
        // (a first row that made no update, or restarted, leaves no whole step)
        __syncthreads();
        if (tid < 3 && static_cast<long long>(clk[2]) > 0) atomicAdd(a.clocks + tid, clk[tid]);
    }
}

template __global__ void k_row_solve<float, true, true, false>(RowArgs<float>);
template __global__ void k_row_solve<float, true, false, false>(RowArgs<float>);
template __global__ void k_row_solve<float, false, true, false>(RowArgs<float>);
template __global__ void k_row_solve<float, false, false, false>(RowArgs<float>);
template __global__ void k_row_solve<float, true, true, true>(RowArgs<float>);
template __global__ void k_row_solve<float, true, false, true>(RowArgs<float>);
template __global__ void k_row_solve<float, false, true, true>(RowArgs<float>);
template __global__ void k_row_solve<float, false, false, true>(RowArgs<float>);
template __global__ void k_row_solve<double, true, true, false>(RowArgs<double>);
template __global__ void k_row_solve<double, true, false, false>(RowArgs<double>);
template __global__ void k_row_solve<double, false, true, false>(RowArgs<double>);
template __global__ void k_row_solve<double, false, false, false>(RowArgs<double>);
template __global__ void k_row_solve<double, true, true, true>(RowArgs<double>);
template __global__ void k_row_solve<double, true, false, true>(RowArgs<double>);
template __global__ void k_row_solve<double, false, true, true>(RowArgs<double>);
template __global__ void k_row_solve<double, false, false, true>(RowArgs<double>);

}  // namespace g2g
