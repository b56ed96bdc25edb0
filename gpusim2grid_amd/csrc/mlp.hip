// Learned warm start: the MLP's training and inference kernels (gfx950).
//
// A 3-layer MLP (in -> hidden -> hidden -> out, GELU) maps a row's per-bus
// injections (and outage mask) to its voltage angles and magnitudes.  Every
// product runs on the bf16 matrix cores with fp32 accumulation
// (v_mfma_f32_32x32x16_bf16) in one form, C = A B^T with both operands
// K-contiguous: whoever writes an activation, a gradient or a weight writes
// the transpose that the other products read beside it, into rows padded to 8
// (zeros), so no product transposes on the way in and any width takes the
// wide loads.  Weights are fp32 (Adam state) with bf16 copies the products read.
//
// The gpusim2grid reference has no learned component; this follows the
// model the reference's paper benchmarks time as "PFdelta" MLPs
// (20260831_neurips_paper/scripts/README.md, ml_injection.py) only in kind.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "mlp.hpp"

namespace g2g {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kBM = 128, kBN = 128, kBK = 32;
constexpr int kPadK = kBK + 8;  // LDS row pitch (bf16): 80 bytes, spreads the 16-byte reads over banks

__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }

__device__ __forceinline__ float gelu_grad(float x)
{
    const float cdf = 0.5f * (1.0f + erff(x * 0.70710678118654752f));
    const float pdf = 0.39894228040143268f * expf(-0.5f * x * x);
    return cdf + x * pdf;
}

// A (M x K) and B (K x N) tiles of one K step, staged k-contiguous in LDS:
// sA[m][k], sB[n][k].
template <bool TA, bool TB>
__device__ __forceinline__ void load_tiles(const GemmArgs& g, int m0, int n0, int k0, __bf16 (*sA)[kPadK],
                                           __bf16 (*sB)[kPadK])
{
    const int t = threadIdx.x;  // 256 threads
    const __bf16 zero = static_cast<__bf16>(0.0f);
    // ---- A: 128 x 32 ------------------------------------------------------
    if (!TA) {  // element (m, k) at A[m * lda + k]
        const int m = t >> 1, kh = (t & 1) * 16;
        const int gm = m0 + m, gk = k0 + kh;
        const __bf16* src = g.A + static_cast<long long>(gm) * g.lda + gk;
        if (gm < g.M && gk + 16 <= g.K && (reinterpret_cast<uintptr_t>(src) & 15) == 0) {
            const u32x4 v0 = reinterpret_cast<const u32x4*>(src)[0];
            const u32x4 v1 = reinterpret_cast<const u32x4*>(src)[1];
            *reinterpret_cast<u32x4*>(&sA[m][kh]) = v0;
            *reinterpret_cast<u32x4*>(&sA[m][kh + 8]) = v1;
        } else {
            for (int i = 0; i < 16; ++i) sA[m][kh + i] = (gm < g.M && gk + i < g.K) ? src[i] : zero;
        }
    } else {  // element (m, k) at A[k * lda + m]
        const int k = t >> 3, mh = (t & 7) * 16;
        const int gk = k0 + k, gm = m0 + mh;
        const __bf16* src = g.A + static_cast<long long>(gk) * g.lda + gm;
        for (int i = 0; i < 16; ++i) sA[mh + i][k] = (gk < g.K && gm + i < g.M) ? src[i] : zero;
    }
    // ---- B: 32 x 128 ------------------------------------------------------
    if (TB) {  // element (k, n) at B[n * ldb + k]
        const int n = t >> 1, kh = (t & 1) * 16;
        const int gn = n0 + n, gk = k0 + kh;
        const __bf16* src = g.B + static_cast<long long>(gn) * g.ldb + gk;
        if (gn < g.N && gk + 16 <= g.K && (reinterpret_cast<uintptr_t>(src) & 15) == 0) {
            const u32x4 v0 = reinterpret_cast<const u32x4*>(src)[0];
            const u32x4 v1 = reinterpret_cast<const u32x4*>(src)[1];
            *reinterpret_cast<u32x4*>(&sB[n][kh]) = v0;
            *reinterpret_cast<u32x4*>(&sB[n][kh + 8]) = v1;
        } else {
            for (int i = 0; i < 16; ++i) sB[n][kh + i] = (gn < g.N && gk + i < g.K) ? src[i] : zero;
        }
    } else {  // element (k, n) at B[k * ldb + n]
        const int k = t >> 3, nh = (t & 7) * 16;
        const int gk = k0 + k, gn = n0 + nh;
        const __bf16* src = g.B + static_cast<long long>(gk) * g.ldb + gn;
        for (int i = 0; i < 16; ++i) sB[nh + i][k] = (gk < g.K && gn + i < g.N) ? src[i] : zero;
    }
}

// C = op(A) op(B) of any layout and alignment (the product entry point's
// general case): 128 x 128 output tile per workgroup of 4 waves (each 64 x 64 as
// 2 x 2 MFMA 32 x 32 tiles), K in steps of 32 through LDS.
template <bool TA, bool TB>
__global__ __launch_bounds__(256) void k_gemm(GemmArgs g)
{
    __shared__ __align__(16) __bf16 sA[kBM][kPadK];
    __shared__ __align__(16) __bf16 sB[kBN][kPadK];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int m0 = blockIdx.y * kBM, n0 = blockIdx.x * kBN;
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    const int lr = lane & 31, lk = (lane >> 5) * 8;
    for (int k0 = 0; k0 < g.K; k0 += kBK) {
        load_tiles<TA, TB>(g, m0, n0, k0, sA, sB);
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < kBK; kk += 16) {
            bf16x8 fa[2], fb[2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
                fa[i] = *reinterpret_cast<const bf16x8*>(&sA[wm * 64 + i * 32 + lr][kk + lk]);
#pragma unroll
            for (int j = 0; j < 2; ++j)
                fb[j] = *reinterpret_cast<const bf16x8*>(&sB[wn * 64 + j * 32 + lr][kk + lk]);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }
    // lane holds column lane % 32 and rows 8 (r / 4) + 4 (lane / 32) + r % 4
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = m0 + wm * 64 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                const int n = n0 + wn * 64 + j * 32 + lr;
                if (m < g.M && n < g.N) g.C[static_cast<long long>(m) * g.ldc + n] = acc[i][j][r];
            }
}

// One 32 x 32 block of a product at (mb, nb): lane holds column lane % 32 and
// rows 8 (r / 4) + 4 (lane / 32) + r % 4, so four consecutive rows of a column,
// one 8-byte store of the transpose.  sq collects the lane's sum of squares.
template <int EPI>
__device__ __forceinline__ void gemm_epilogue(const GemmArgs& g, int mb, int nb, const f32x16& v, float& sq)
{
    const int lane = threadIdx.x & 63;
    const int n = nb + (lane & 31), m0 = mb + 4 * (lane >> 5);
    const bool cols = n < g.N;
    float col = 0.0f;
    const float bias = (EPI == kEpiBiasF32 || EPI == kEpiGelu || EPI == kEpiMse) && cols ? g.bias[n] : 0.0f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int mq = m0 + 8 * q;
        __bf16 h[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int m = mq + s;
            const bool in = cols && m < g.M;
            const long long mc = m;
            const float x = v[4 * q + s];
            float y = 0.0f;
            if (EPI == kEpiF32) {
                if (in) g.C[mc * g.ldc + n] = x;
            } else if (EPI == kEpiBiasF32) {
                if (in) g.C[mc * g.ldc + n] = x + bias;
            } else if (EPI == kEpiGrad) {
                if (in) {
                    g.C[mc * g.ldc + n] = x;
                    sq = fmaf(x, x, sq);
                }
            } else if (EPI == kEpiGelu) {
                const float z = x + bias;
                if (in && g.Z) g.Z[mc * g.ldz + n] = z;
                y = in ? gelu(z) : 0.0f;
            } else if (EPI == kEpiGeluBwd) {
                y = in ? x * gelu_grad(g.Z[mc * g.ldz + n]) : 0.0f;
                col += y;
            } else {  // kEpiMse
                const float d = in ? x + bias - g.T[mc * g.ldc + n] : 0.0f;
                sq = fmaf(d, d, sq);
                y = 2.0f * g.scale * d;
                col += y;
            }
            if (EPI == kEpiGelu || EPI == kEpiGeluBwd || EPI == kEpiMse) {
                h[s] = static_cast<__bf16>(y);
                if (in && g.H) g.H[mc * g.ldh + n] = h[s];
            }
        }
        if (EPI == kEpiGelu || EPI == kEpiGeluBwd || EPI == kEpiMse) {
            if (g.Ht && cols && mq < g.Mt) {
                uint2 w;
                __builtin_memcpy(&w, h, sizeof(w));
                *reinterpret_cast<uint2*>(g.Ht + static_cast<long long>(n) * g.Mt + mq) = w;
            }
        }
    }
    if (EPI == kEpiGeluBwd || EPI == kEpiMse) {
        col += __shfl_xor(col, 32, 64);
        if (lane < 32 && cols && mb < g.M) g.colsum[static_cast<long long>(mb / 32) * g.N + n] = col;
    }
}

__device__ __forceinline__ float wave_sum(float x)
{
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    return x;
}

// C = A B^T: 128 x 128 output tile per workgroup of 4 waves (each 64 x 64 as
// 2 x 2 MFMA 32x32x16 tiles); K in steps of 64 through a double-buffered LDS
// stage, the next step's global loads in flight while the current one is
// multiplied.  A product with few tiles and a long K (512 x 1,024 outputs over
// 13,000 inputs: 32 tiles) is split over gridDim.z, the partial sums added in
// split order by k_gemm_sum (unsplit on 32 of 256 CUs: about 270 us; split by 8: 45 + 9 us).
constexpr int kFK = 64, kFPad = 8;

__device__ __forceinline__ void kc_load(const __bf16* base, long long ld, int rows, int r0, int k0, int K, int t,
                                        u32x4 (&reg)[4])
{
    const int kc = (t & 7) * 8;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = r0 + (t >> 3) + 32 * i;
        const int k = k0 + kc;
        if (r < rows && k < K) reg[i] = *reinterpret_cast<const u32x4*>(base + static_cast<long long>(r) * ld + k);
        else reg[i] = u32x4{0u, 0u, 0u, 0u};
    }
}

__device__ __forceinline__ void kc_store(__bf16 (*s)[kFK + kFPad], int t, const u32x4 (&reg)[4])
{
    const int kc = (t & 7) * 8;
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<u32x4*>(&s[(t >> 3) + 32 * i][kc]) = reg[i];
}

template <int EPI>
__global__ __launch_bounds__(256) void k_gemm_kc(GemmArgs g)
{
    __shared__ __align__(16) __bf16 sA[2][kBM][kFK + kFPad];
    __shared__ __align__(16) __bf16 sB[2][kBN][kFK + kFPad];
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = t >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int m0 = blockIdx.y * kBM, n0 = blockIdx.x * kBN;
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    const int lr = lane & 31, lk = (lane >> 5) * 8;
    u32x4 ra[4], rb[4];
    int kb = 0, ke = g.K;
    if (EPI == kEpiF32 && g.k_split > 0) {
        kb = static_cast<int>(blockIdx.z) * g.k_split;
        ke = min(kb + g.k_split, g.K);
        g.C += static_cast<long long>(blockIdx.z) * g.M * g.N;
    }
    kc_load(g.A, g.lda, g.M, m0, kb, ke, t, ra);
    kc_load(g.B, g.ldb, g.N, n0, kb, ke, t, rb);
    kc_store(sA[0], t, ra);
    kc_store(sB[0], t, rb);
    __syncthreads();
    int cur = 0;
    for (int k0 = kb; k0 < ke; k0 += kFK) {
        const bool more = k0 + kFK < ke;
        if (more) {
            kc_load(g.A, g.lda, g.M, m0, k0 + kFK, ke, t, ra);
            kc_load(g.B, g.ldb, g.N, n0, k0 + kFK, ke, t, rb);
        }
#pragma unroll
        for (int kk = 0; kk < kFK; kk += 16) {
            bf16x8 fa[2], fb[2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
                fa[i] = *reinterpret_cast<const bf16x8*>(&sA[cur][wm * 64 + i * 32 + lr][kk + lk]);
#pragma unroll
            for (int j = 0; j < 2; ++j)
                fb[j] = *reinterpret_cast<const bf16x8*>(&sB[cur][wn * 64 + j * 32 + lr][kk + lk]);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
        }
        if (more) {
            kc_store(sA[cur ^ 1], t, ra);
            kc_store(sB[cur ^ 1], t, rb);
        }
        __syncthreads();
        cur ^= 1;
    }
    float sq = 0.0f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
            gemm_epilogue<EPI>(g, m0 + wm * 64 + i * 32, n0 + wn * 64 + j * 32, acc[i][j], sq);
    if (EPI == kEpiGrad || EPI == kEpiMse) {
        sq = wave_sum(sq);
        if (lane == 0) g.sums[(blockIdx.y * gridDim.x + blockIdx.x) * 4 + wave] = sq;
    }
}

// a split product's sum and epilogue: one wave per 32 x 32 outputs (a split
// product has few of them, so one per workgroup)
template <int EPI>
__global__ __launch_bounds__(64) void k_gemm_sum(GemmArgs g, const float* __restrict__ part, int splits)
{
    const int lane = threadIdx.x;
    const int mb = blockIdx.y * 32, nb = blockIdx.x * 32;
    const int n = nb + (lane & 31);
    const long long mn = static_cast<long long>(g.M) * g.N;
    // every output's split is loaded before any is added: 16 loads in flight
    f32x16 v;
    long long at[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int m = mb + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        at[r] = static_cast<long long>(m < g.M ? m : 0) * g.N + (n < g.N ? n : 0);
        v[r] = part[at[r]];
    }
    for (int s = 1; s < splits; ++s) {
        const float* p = part + s * mn;
        float x[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = p[at[r]];
#pragma unroll
        for (int r = 0; r < 16; ++r) v[r] += x[r];
    }
    float sq = 0.0f;
    gemm_epilogue<EPI>(g, mb, nb, v, sq);
    if (EPI == kEpiGrad || EPI == kEpiMse) {
        sq = wave_sum(sq);
        if (lane == 0) g.sums[blockIdx.y * gridDim.x + blockIdx.x] = sq;
    }
}

// a 64 x 64 bf16 tile in LDS: [k][n], written out as rows n of 64 consecutive k
constexpr int kTT = 64, kTPitch = kTT + 2;
__device__ __forceinline__ void store_transposed(const __bf16 (*tile)[kTPitch], int k0, int n0, int K, int N,
                                                 __bf16* Wt, long long ldt)
{
    // 16-byte chunks of 8 k; rows are padded to a multiple of 8 (the tile holds zeros past K)
    for (int c = threadIdx.x; c < kTT * kTT / 8; c += 256) {
        const int n = c / (kTT / 8), k = (c % (kTT / 8)) * 8;
        if (n0 + n >= N || k0 + k >= (K + 7) / 8 * 8) continue;
        __bf16 h[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) h[i] = tile[k + i][n];
        u32x4 w;
        __builtin_memcpy(&w, h, sizeof(w));
        *reinterpret_cast<u32x4*>(Wt + static_cast<long long>(n0 + n) * ldt + k0 + k) = w;
    }
}

__device__ __forceinline__ float adam(float& w, float& m, float& v, float g, const AdamArgs& a, float gs)
{
    const float gi = g * gs;
    const float mi = a.b1 * m + (1.0f - a.b1) * gi;
    const float vi = a.b2 * v + (1.0f - a.b2) * gi * gi;
    m = mi;
    v = vi;
    w = w - a.lr * (mi * a.c1) / (sqrtf(vi * a.c2) + a.eps);
    return w;
}

// min(1, clip / ||g||)
__device__ __forceinline__ float grad_scale(const AdamArgs& a)
{
    if (!a.gnorm2) return 1.0f;
    const float nrm = sqrtf(*a.gnorm2);
    return nrm > a.clip ? a.clip / nrm : 1.0f;
}

// Bound by HBM: 28 bytes a weight of fp32 state and 2 - 4 of copies; the
// transposed copy goes through LDS here instead of a pass of its own that
// reads the weights again (59 us of a 6,500-bus step).
__global__ __launch_bounds__(256) void k_weights(float* __restrict__ w, float* __restrict__ m, float* __restrict__ v,
                                                 const float* __restrict__ g, int K, int N, AdamArgs a,
                                                 __bf16* __restrict__ Wt, long long ldt, __bf16* __restrict__ Wn,
                                                 long long ldn)
{
    __shared__ __bf16 tile[kTT][kTPitch];
    const int k0 = blockIdx.y * kTT, n0 = blockIdx.x * kTT;
    const int c = (threadIdx.x & 15) * 4, r = threadIdx.x >> 4;
    const float gs = m ? grad_scale(a) : 1.0f;
    const bool wide = (N & 3) == 0;  // rows and matrices start 16-byte aligned
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int k = k0 + r + 16 * i, n = n0 + c;
        float x[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        const long long at = static_cast<long long>(k) * N + n;
        if (k < K && wide && n < N) {
            float4 w4 = *reinterpret_cast<const float4*>(w + at);
            if (m) {
                float4 m4 = *reinterpret_cast<const float4*>(m + at), v4 = *reinterpret_cast<const float4*>(v + at);
                const float4 g4 = *reinterpret_cast<const float4*>(g + at);
                adam(w4.x, m4.x, v4.x, g4.x, a, gs);
                adam(w4.y, m4.y, v4.y, g4.y, a, gs);
                adam(w4.z, m4.z, v4.z, g4.z, a, gs);
                adam(w4.w, m4.w, v4.w, g4.w, a, gs);
                *reinterpret_cast<float4*>(w + at) = w4;
                *reinterpret_cast<float4*>(m + at) = m4;
                *reinterpret_cast<float4*>(v + at) = v4;
            }
            x[0] = w4.x;
            x[1] = w4.y;
            x[2] = w4.z;
            x[3] = w4.w;
        } else if (k < K) {
            for (int j = 0; j < 4 && n + j < N; ++j) {
                float wj = w[at + j];
                if (m) {
                    float mj = m[at + j], vj = v[at + j];
                    adam(wj, mj, vj, g[at + j], a, gs);
                    w[at + j] = wj;
                    m[at + j] = mj;
                    v[at + j] = vj;
                }
                x[j] = wj;
            }
        }
        __bf16 h[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            h[j] = static_cast<__bf16>(x[j]);
            tile[r + 16 * i][c + j] = h[j];
        }
        if (Wn && k < K && n < ldn) {  // (ldn a multiple of 8: pads get their zeros)
            uint2 p;
            __builtin_memcpy(&p, h, sizeof(p));
            *reinterpret_cast<uint2*>(Wn + static_cast<long long>(k) * ldn + n) = p;
        }
    }
    __syncthreads();
    store_transposed(tile, k0, n0, K, N, Wt, ldt);
}

__global__ __launch_bounds__(256) void k_adam_bias(float* __restrict__ w, float* __restrict__ m,
                                                   float* __restrict__ v, const float* __restrict__ g, BiasSegs s,
                                                   AdamArgs a)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    const float gs = grad_scale(a);
    for (int q = 0; q < 3; ++q) {
        if (i < s.len[q]) {
            const long long at = s.off[q] + i;
            adam(w[at], m[at], v[at], g[at], a, gs);
            return;
        }
        i -= s.len[q];
    }
}

__global__ __launch_bounds__(256) void k_bias_grad(BiasGradArgs a)
{
    __shared__ float part[4];
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    float x = 0.0f;
    for (int q = 0; q < 3; ++q) {
        if (i >= 0 && i < a.s.len[q]) {
            for (int r = 0; r < a.rows; ++r) x += a.colsum[q][static_cast<long long>(r) * a.s.len[q] + i];
            a.g[a.s.off[q] + i] = x;
        }
        i -= a.s.len[q];
    }
    const float sq = wave_sum(x * x);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = sq;
    __syncthreads();
    if (threadIdx.x == 0) a.sums[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

__global__ __launch_bounds__(1024) void k_finish(const float* __restrict__ a, int na, float scale,
                                                 const float* __restrict__ b, int nb, float* __restrict__ loss,
                                                 float* __restrict__ gnorm2)
{
    __shared__ float sa[16], sb[16];
    float x = 0.0f, y = 0.0f;
    for (int i = threadIdx.x; i < na; i += 1024) x += a[i];
    for (int i = threadIdx.x; i < nb; i += 1024) y += b[i];
    x = wave_sum(x);
    y = wave_sum(y);
    if ((threadIdx.x & 63) == 0) {
        sa[threadIdx.x >> 6] = x;
        sb[threadIdx.x >> 6] = y;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < 16; ++i) {
            x += sa[i];
            y += sb[i];
        }
        *loss = scale * x;
        *gnorm2 = y;
    }
}

__global__ __launch_bounds__(256) void k_stage_x(const float* __restrict__ X, int M, int n, __bf16* __restrict__ Xb,
                                                 long long ldx, __bf16* __restrict__ Xt, int Mt)
{
    __shared__ __bf16 tile[kTT][kTPitch];
    const int m0 = blockIdx.y * kTT, n0 = blockIdx.x * kTT;
    const int c = (threadIdx.x & 15) * 4, r = threadIdx.x >> 4;
    const bool wide = (n & 3) == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + r + 16 * i, k = n0 + c;
        float x[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (m < M && wide && k < n) {
            const float4 q = *reinterpret_cast<const float4*>(X + static_cast<long long>(m) * n + k);
            x[0] = q.x;
            x[1] = q.y;
            x[2] = q.z;
            x[3] = q.w;
        } else if (m < M) {
            for (int j = 0; j < 4 && k + j < n; ++j) x[j] = X[static_cast<long long>(m) * n + k + j];
        }
        __bf16 h[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            h[j] = static_cast<__bf16>(x[j]);
            tile[r + 16 * i][c + j] = h[j];
        }
        if (m < M && k < ldx) {
            uint2 p;
            __builtin_memcpy(&p, h, sizeof(p));
            *reinterpret_cast<uint2*>(Xb + static_cast<long long>(m) * ldx + k) = p;
        }
    }
    if (!Xt) return;
    __syncthreads();
    store_transposed(tile, m0, n0, M, n, Xt, Mt);
}

// Features and start voltages in the batch's tiled layout, [row / 64][bus][row % 64]:
//   features: per bus (P - mu) / sigma, (Q - mu) / sigma, then the optional
//             0/1 outage mask -> bf16 [M][F];
//   start V:  V = Vm exp(j Va) from the network output Y (normalised Va, Vm
//             per bus), Vm held at the set-point where it is fixed (PV, slack)
//             and Va = 0 at the slack.
// Both sides are coalesced: a block moves a patch
// of one tile's 64 rows by 32 buses through LDS (the tiled side is read or
// written 64 lanes = 1 KB at a time, the row-major side 64 features of a row
// at a time).  Grid: (ceil(n / 32), ceil(M / 64)), 256 threads.
__global__ __launch_bounds__(256) void k_features_tiles_t(const double2* __restrict__ S_tiles, int M, int n,
                                                          const float* __restrict__ mu,
                                                          const float* __restrict__ sigma, __bf16* __restrict__ X,
                                                          long long ldx)
{
    __shared__ double2 sS[kPatchBuses][64];
    const int t = threadIdx.x;
    const int b0 = blockIdx.x * kPatchBuses, tile = blockIdx.y;
    for (int i = t; i < kPatchBuses * 64; i += 256) {
        const int bl = i >> 6, lane = i & 63;
        const int b = b0 + bl;
        sS[bl][lane] = b < n ? S_tiles[(static_cast<long long>(tile) * n + b) * 64 + lane] : make_double2(0.0, 0.0);
    }
    __syncthreads();
    const int rr = t >> 2, q = t & 3;  // row of the patch, quarter of its 64 features
    const int r = tile * 64 + rr;
    if (r >= M) return;
    __bf16* x = X + static_cast<long long>(r) * ldx;
    constexpr int kQ = kPatchBuses / 4;  // buses of this thread: 2 kQ contiguous features
    const int bq = b0 + q * kQ;
    if (bq + kQ <= n && (ldx & 7) == 0) {
        // the 2 kQ features as 16-byte stores (row starts and bq are 16-byte aligned)
        __bf16 o[2 * kQ];
#pragma unroll
        for (int k = 0; k < kQ; ++k) {
            const int b = bq + k;
            const double2 v = sS[q * kQ + k][rr];
            o[2 * k] = static_cast<__bf16>(static_cast<float>((v.x - mu[2 * b]) / sigma[2 * b]));
            o[2 * k + 1] = static_cast<__bf16>(static_cast<float>((v.y - mu[2 * b + 1]) / sigma[2 * b + 1]));
        }
        uint4 w[2 * kQ * sizeof(__bf16) / sizeof(uint4)];
        __builtin_memcpy(w, o, sizeof(o));
        uint4* dst = reinterpret_cast<uint4*>(x + 2 * bq);
#pragma unroll
        for (int i = 0; i < static_cast<int>(sizeof(w) / sizeof(uint4)); ++i) dst[i] = w[i];
        return;
    }
    for (int k = 0; k < kQ; ++k) {
        const int bl = q * kQ + k;
        const int b = b0 + bl;
        if (b >= n) break;
        const double2 v = sS[bl][rr];
        x[2 * b] = static_cast<__bf16>(static_cast<float>((v.x - mu[2 * b]) / sigma[2 * b]));
        x[2 * b + 1] = static_cast<__bf16>(static_cast<float>((v.y - mu[2 * b + 1]) / sigma[2 * b + 1]));
    }
}

// outage-mask features 2n .. 2n + n_mask of each row
__global__ void k_mask_features(const unsigned char* __restrict__ mask, int M, int n, int n_mask,
                                __bf16* __restrict__ X, long long ldx)
{
    const long long gid = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (gid >= static_cast<long long>(M) * n_mask) return;
    const int r = static_cast<int>(gid / n_mask);
    const int m = static_cast<int>(gid - static_cast<long long>(r) * n_mask);
    X[static_cast<long long>(r) * ldx + 2 * n + m] = static_cast<__bf16>(static_cast<float>(mask[gid]));
}

__global__ __launch_bounds__(256) void k_warm_v_tiles_t(const float* __restrict__ Y, long long ldy, int M, int n,
                                                        const float* __restrict__ mu,
                                                        const float* __restrict__ sigma,
                                                        const double* __restrict__ vfix, const int* __restrict__ kind,
                                                        double2* __restrict__ V_tiles)
{
    __shared__ float2 sY[kPatchBuses][64];
    const int t = threadIdx.x;
    const int b0 = blockIdx.x * kPatchBuses, tile = blockIdx.y;
    {
        const int rr = t >> 2, q = t & 3;
        const int r = tile * 64 + rr;
        const float* y = Y + static_cast<long long>(r) * ldy;
        constexpr int kQ = kPatchBuses / 4;  // buses of this thread: 2 kQ contiguous outputs
        const int bq = b0 + q * kQ;
        if (r < M && bq + kQ <= n && (ldy & 3) == 0) {
            // 16-byte loads (row starts and bq are 16-byte aligned)
            const float4* src = reinterpret_cast<const float4*>(y + 2 * bq);
#pragma unroll
            for (int k = 0; k < kQ / 2; ++k) {
                const float4 f = src[k];
                sY[q * kQ + 2 * k][rr] = make_float2(f.x, f.y);
                sY[q * kQ + 2 * k + 1][rr] = make_float2(f.z, f.w);
            }
        } else {
            for (int k = 0; k < kQ; ++k) {
                const int bl = q * kQ + k;
                const int b = b0 + bl;
                sY[bl][rr] = (r < M && b < n) ? make_float2(y[2 * b], y[2 * b + 1]) : make_float2(0.f, 0.f);
            }
        }
    }
    __syncthreads();
    for (int i = t; i < kPatchBuses * 64; i += 256) {
        const int bl = i >> 6, lane = i & 63;
        const int b = b0 + bl, r = tile * 64 + lane;
        if (b >= n || r >= M) continue;
        if (kind[b] == 2) continue;  // a fixed bus keeps the row's start V
        const float2 o = sY[bl][lane];
        double va = static_cast<double>(o.x) * sigma[2 * b] + mu[2 * b];
        double vm = static_cast<double>(o.y) * sigma[2 * b + 1] + mu[2 * b + 1];
        if (kind[b] != 1) vm = vfix[b];
        double sn, cs;
        sincos(va, &sn, &cs);
        V_tiles[(static_cast<long long>(tile) * n + b) * 64 + lane] = make_double2(vm * cs, vm * sn);
    }
}

template __global__ void k_gemm_kc<kEpiF32>(GemmArgs);
template __global__ void k_gemm_kc<kEpiBiasF32>(GemmArgs);
template __global__ void k_gemm_kc<kEpiGelu>(GemmArgs);
template __global__ void k_gemm_kc<kEpiGeluBwd>(GemmArgs);
template __global__ void k_gemm_kc<kEpiMse>(GemmArgs);
template __global__ void k_gemm_kc<kEpiGrad>(GemmArgs);
template __global__ void k_gemm_sum<kEpiBiasF32>(GemmArgs, const float*, int);
template __global__ void k_gemm_sum<kEpiGelu>(GemmArgs, const float*, int);
template __global__ void k_gemm_sum<kEpiGeluBwd>(GemmArgs, const float*, int);
template __global__ void k_gemm_sum<kEpiMse>(GemmArgs, const float*, int);
template __global__ void k_gemm_sum<kEpiGrad>(GemmArgs, const float*, int);
template __global__ void k_gemm<false, false>(GemmArgs);
template __global__ void k_gemm<false, true>(GemmArgs);
template __global__ void k_gemm<true, false>(GemmArgs);
template __global__ void k_gemm<true, true>(GemmArgs);

}  // namespace g2g
