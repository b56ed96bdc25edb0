// MLP warm start: kernel interfaces shared by mlp.hip and the C ABI.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace g2g {

enum GemmEpilogue : int {
    kEpiF32 = 0,      // C = A B^T (a split's partial sums included)
    kEpiBiasF32 = 1,  // C = A B^T + bias
    kEpiGelu = 2,     // z = A B^T + bias: Z (fp32, nullable), H and its transpose = gelu(z)
    kEpiGeluBwd = 3,  // dz = (A B^T) gelu'(Z): H (nullable), its transpose, column sums
    kEpiMse = 4,      // d = A B^T + bias - T: H and its transpose = 2 scale d, column sums, sum of d^2
    kEpiGrad = 5,     // C = A B^T, sum of squares
};

// C = A B^T with both operands K-contiguous: A M x K (row m at A + m lda), B
// N x K (row n at B + n ldb), 16-byte aligned rows, K a multiple of 8.
struct GemmArgs {
    const __bf16* A;
    long long lda;
    const __bf16* B;
    long long ldb;
    int M, N, K;
    int k_split;        // > 0: split s of gridDim.z sums [s k_split, (s + 1) k_split), its partial at C + s M N
    float* C;
    long long ldc;
    __bf16* H;          // M x N, pitch ldh
    long long ldh;
    __bf16* Ht;         // N x Mt (nullable), rows of Mt: columns m >= M are written as 0
    int Mt;
    float* Z;
    long long ldz;
    const float* bias;
    const float* T;     // targets, pitch ldc
    float scale;
    float* colsum;      // [ceil(M / 32)][N] column sums of 32 rows
    float* sums;        // one per wavefront of the launch: sum of squares (kEpiGrad, kEpiMse)
};

template <bool TA, bool TB>
__global__ void k_gemm(GemmArgs g);
template <int EPI>
__global__ void k_gemm_kc(GemmArgs g);
// the epilogue of a split product: part [splits][M][N]
template <int EPI>
__global__ void k_gemm_sum(GemmArgs g, const float* part, int splits);

// Adam's constants of a step; gnorm2 (nullable) is the gradient's squared
// norm, which scales it by min(1, clip / ||g||)
struct AdamArgs {
    float lr, b1, b2, eps, c1, c2;
    const float* gnorm2;
    float clip;
};
// One weight matrix (K x N, fp32 row-major) and its bf16 copies: Wt (N x ldt,
// transposed) and Wn (K x ldn, nullable).  With m: an Adam step first.
__global__ void k_weights(float* w, float* m, float* v, const float* g, int K, int N, AdamArgs a, __bf16* Wt,
                          long long ldt, __bf16* Wn, long long ldn);
// the biases' Adam step: three segments {offset, length}
struct BiasSegs {
    long long off[3];
    int len[3];
};
__global__ void k_adam_bias(float* w, float* m, float* v, const float* g, BiasSegs s, AdamArgs a);
// the biases' gradients from the products' column sums [rows[i]][len[i]], and
// each block's sum of their squares
struct BiasGradArgs {
    BiasSegs s;
    const float* colsum[3];
    int rows;
    float* g;
    float* sums;
};
__global__ void k_bias_grad(BiasGradArgs a);
// out[0] = scale x the sum of a [0, na), out[1] = the sum of b [0, nb)
__global__ void k_finish(const float* a, int na, float scale, const float* b, int nb, float* loss, float* gnorm2);
// X (fp32, M x n) -> bf16 rows of pitch ldx and (nullable) their transpose, rows of Mt
__global__ void k_stage_x(const float* X, int M, int n, __bf16* Xb, long long ldx, __bf16* Xt, int Mt);
__global__ void k_fill_int(int* p, int v, long long n);
constexpr int kPatchBuses = 32;  // buses per block of the tiled-layout conversions
__global__ void k_features_tiles_t(const double2* S_tiles, int M, int n, const float* mu, const float* sigma,
                                   __bf16* X, long long ldx);
__global__ void k_mask_features(const unsigned char* mask, int M, int n, int n_mask, __bf16* X, long long ldx);
__global__ void k_warm_v_tiles_t(const float* Y, long long ldy, int M, int n, const float* mu, const float* sigma,
                                 const double* vfix, const int* kind, double2* V_tiles);

}  // namespace g2g
