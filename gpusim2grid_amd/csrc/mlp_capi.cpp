// C ABI of the learned warm start (see include/gpusim2grid_amd.h).
#include <hip/hip_runtime.h>

#include <algorithm>

#include <cmath>
#include <cstring>
#include <memory>
#include <random>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/gpusim2grid_amd.h"
#include "capi_common.hpp"
#include "mlp.hpp"

using namespace g2g;

struct g2g_mlp_s {
    int n_in = 0, H = 0, n_out = 0;
    hipStream_t stream = nullptr;
    // fp32 parameters, contiguous: W1 [n_in x H], b1 [H], W2 [H x H], b2 [H], W3 [H x n_out], b3 [n_out]
    size_t o_W1 = 0, o_b1 = 0, o_W2 = 0, o_b2 = 0, o_W3 = 0, o_b3 = 0, n_params = 0;
    float* w = nullptr;
    float* m = nullptr;
    float* v = nullptr;
    float* g = nullptr;
    // bf16 copies the products read, rows K-contiguous and padded to 8: the
    // transposed weights (forward) and, of the upper layers, the weights as
    // they are (backward)
    __bf16 *W1t = nullptr, *W2t = nullptr, *W3t = nullptr, *W2n = nullptr, *W3n = nullptr;
    int step = 0;
    // normalisation (features: z-score per input; outputs: per output)
    float* in_mu = nullptr;
    float* in_sigma = nullptr;
    float* out_mu = nullptr;
    float* out_sigma = nullptr;
    // buses for the warm start: kind (0 pv, 1 pq, 2 fixed), |V| of pv buses
    int* kind = nullptr;
    double* vfix = nullptr;
    int n_bus = 0;
    // workspace of M rows: activations (rows padded to 8) ...
    int ws_M = 0;
    __bf16 *X = nullptr, *H1 = nullptr, *H2 = nullptr;
    float* Y = nullptr;
    // ... and of a training step: pre-activations, transposes (rows of M
    // padded to 8), gradients, column sums of 32 rows, sums of squares
    int tr_M = 0;
    float *Z1 = nullptr, *Z2 = nullptr, *T = nullptr;
    __bf16 *Xt = nullptr, *H1t = nullptr, *H2t = nullptr, *dYb = nullptr, *dYt = nullptr, *dZ2b = nullptr, *dZ2t = nullptr,
           *dZ1t = nullptr;
    float *cs1 = nullptr, *cs2 = nullptr, *cs3 = nullptr, *sums = nullptr, *loss_sums = nullptr;
    // partial sums of split products (grown on use)
    float* part = nullptr;
    size_t part_cap = 0;
    float* loss = nullptr;
    float clip = 0.0f;          // gradient-norm clip of the training steps (0: off)
    DeviceScratch ws, tr, pt;  // workspace buffers (freed on growth / destruction)
    DeviceScratch own;         // parameters and state

    static int pad8(int n) { return (n + 7) / 8 * 8; }
    int kin() const { return pad8(n_in); }
    int kh() const { return pad8(H); }
    int kout() const { return pad8(n_out); }

    // the bf16 copies from the fp32 masters, after an Adam step (a) or without
    void refresh_weights(hipStream_t st, const AdamArgs* a)
    {
        auto layer = [&](size_t off, int K, int N, __bf16* Wt, long long ldt, __bf16* Wn, long long ldn) {
            const dim3 grid((N + 63) / 64, (K + 63) / 64);
            k_weights<<<grid, 256, 0, st>>>(w + off, a ? m + off : nullptr, v + off, g + off, K, N, a ? *a : AdamArgs{},
                                            Wt, ldt, Wn, ldn);
        };
        layer(o_W1, n_in, H, W1t, kin(), nullptr, 0);
        layer(o_W2, H, H, W2t, kh(), W2n, kh());
        layer(o_W3, H, n_out, W3t, kh(), W3n, kout());
        if (a) {
            const BiasSegs b{{static_cast<long long>(o_b1), static_cast<long long>(o_b2), static_cast<long long>(o_b3)},
                             {H, H, n_out}};
            k_adam_bias<<<blocks_for(2LL * H + n_out, 256), 256, 0, st>>>(w, m, v, g, b, *a);
        }
        HIPCHK(hipGetLastError());
    }

    void workspace(int M)
    {
        if (M <= ws_M) return;
        HIPCHK(hipStreamSynchronize(stream));
        ws.release();
        ws_M = 0;
        const size_t r = static_cast<size_t>(M);
        // (padding columns are zeroed once and never written)
        auto padded = [&](size_t cols, size_t pitch) {
            __bf16* p = ws.get<__bf16>(r * pitch);
            if (cols != pitch) HIPCHK(hipMemsetAsync(p, 0, r * pitch * sizeof(__bf16), stream));
            return p;
        };
        X = padded(n_in, kin());
        H1 = padded(H, kh());
        H2 = padded(H, kh());
        Y = ws.get<float>(r * n_out);
        ws_M = M;
    }

    // waves of a product's launch, at most: 64 x 64 outputs each or (split)
    // 32 x 32, in workgroups of 128 x 128
    static size_t waves(int M, int N)
    {
        return 16 * static_cast<size_t>((M + 127) / 128) * static_cast<size_t>((N + 127) / 128);
    }

    void train_workspace(int M)
    {
        workspace(M);
        if (M <= tr_M) return;
        HIPCHK(hipStreamSynchronize(stream));
        tr.release();
        tr_M = 0;
        const size_t r = static_cast<size_t>(M), mt = static_cast<size_t>(pad8(M)), rb = (r + 31) / 32;
        Z1 = tr.get<float>(r * H);
        Z2 = tr.get<float>(r * H);
        T = tr.get<float>(r * n_out);
        Xt = tr.get<__bf16>(mt * n_in);
        H1t = tr.get<__bf16>(mt * H);
        H2t = tr.get<__bf16>(mt * H);
        dYb = tr.get<__bf16>(r * kout());
        dYt = tr.get<__bf16>(mt * n_out);
        dZ2b = tr.get<__bf16>(r * kh());
        dZ2t = tr.get<__bf16>(mt * H);
        dZ1t = tr.get<__bf16>(mt * H);
        HIPCHK(hipMemsetAsync(dYb, 0, r * kout() * sizeof(__bf16), stream));
        HIPCHK(hipMemsetAsync(dZ2b, 0, r * kh() * sizeof(__bf16), stream));
        cs1 = tr.get<float>(rb * H);
        cs2 = tr.get<float>(rb * H);
        cs3 = tr.get<float>(rb * n_out);
        sums = tr.get<float>(waves(n_in, H) + waves(H, H) + waves(H, n_out) +
                             blocks_for(2LL * H + n_out, 256));
        loss_sums = tr.get<float>(waves(M, n_out));
        if (!loss) loss = own.get<float>(2);
        tr_M = M;
    }

    float* partials(size_t n)
    {
        if (n > part_cap) {
            HIPCHK(hipStreamSynchronize(stream));
            pt.release();
            part_cap = 0;
            part = pt.get<float>(n);
            part_cap = n;
        }
        return part;
    }
};

namespace {

template <bool TA, bool TB>
void gemm(hipStream_t st, const __bf16* A, long long lda, const __bf16* B, long long ldb, int M, int N, int K,
          float* C, long long ldc)
{
    GemmArgs a{};
    a.A = A;
    a.lda = lda;
    a.B = B;
    a.ldb = ldb;
    a.M = M;
    a.N = N;
    a.K = K;
    a.C = C;
    a.ldc = ldc;
    const dim3 grid((N + 127) / 128, (M + 127) / 128);
    k_gemm<TA, TB><<<grid, 256, 0, st>>>(a);
    HIPCHK(hipGetLastError());
}

// X (fp32, M x n_in, host or device) -> the workspace's bf16 X and, for a
// training step, its transpose
void stage_x(g2g_mlp_s* p, const float* X, int M, int on_device, bool train)
{
    const size_t n = static_cast<size_t>(M) * p->n_in;
    const float* src = X;
    DeviceScratch tmp;
    if (!on_device) {
        float* d = tmp.get<float>(n);
        HIPCHK(hipMemcpyAsync(d, X, n * sizeof(float), hipMemcpyHostToDevice, p->stream));
        src = d;
    }
    const dim3 grid((p->n_in + 63) / 64, (M + 63) / 64);
    k_stage_x<<<grid, 256, 0, p->stream>>>(src, M, p->n_in, p->X, p->kin(), train ? p->Xt : nullptr,
                                           g2g_mlp_s::pad8(M));
    HIPCHK(hipGetLastError());
    if (!on_device) HIPCHK(hipStreamSynchronize(p->stream));
}

// C = A B^T (A M x K, B N x K).  Fewer than half a tile per CU: K is split so
// that the launch covers the CUs (at least 256 of K a split), the partials
// summed, in order, by a second launch that runs the epilogue.  Returns the
// floats written to `sums`.
template <int EPI>
size_t product(g2g_mlp_s* p, GemmArgs a)
{
    constexpr int kCus = 256, kMinK = 256;
    const int gx = (a.N + 127) / 128, gy = (a.M + 127) / 128, tiles = gx * gy;
    int splits = tiles >= kCus / 2 ? 1 : std::min(kCus / tiles, a.K / kMinK);
    if (splits <= 1) {
        k_gemm_kc<EPI><<<dim3(gx, gy), 256, 0, p->stream>>>(a);
        HIPCHK(hipGetLastError());
        return 4 * static_cast<size_t>(tiles);
    }
    GemmArgs s = a;
    s.k_split = (((a.K + splits - 1) / splits) + 63) / 64 * 64;
    splits = (a.K + s.k_split - 1) / s.k_split;
    s.C = p->partials(static_cast<size_t>(splits) * a.M * a.N);
    s.ldc = a.N;
    k_gemm_kc<kEpiF32><<<dim3(gx, gy, splits), 256, 0, p->stream>>>(s);
    const dim3 grid((a.N + 31) / 32, (a.M + 31) / 32);
    k_gemm_sum<EPI><<<grid, 64, 0, p->stream>>>(a, s.C, splits);
    HIPCHK(hipGetLastError());
    return static_cast<size_t>(grid.x) * grid.y;
}

GemmArgs operands(const __bf16* A, long long lda, const __bf16* B, long long ldb, int M, int N, int K)
{
    GemmArgs a{};
    a.A = A;
    a.lda = lda;
    a.B = B;
    a.ldb = ldb;
    a.M = M;
    a.N = N;
    a.K = K;
    return a;
}

// the hidden layers of the staged X; train: with the pre-activations and
// transposes the backward pass needs
void hidden(g2g_mlp_s* p, int M, bool train)
{
    const int mt = g2g_mlp_s::pad8(M);
    auto layer = [&](const __bf16* A, int ka, const __bf16* Wt, size_t o_b, __bf16* Hh, __bf16* Ht, float* Z) {
        GemmArgs a = operands(A, ka, Wt, ka, M, p->H, ka);
        a.bias = p->w + o_b;
        a.H = Hh;
        a.ldh = p->kh();
        a.Ht = train ? Ht : nullptr;
        a.Mt = mt;
        a.Z = train ? Z : nullptr;
        a.ldz = p->H;
        product<kEpiGelu>(p, a);
    };
    layer(p->X, p->kin(), p->W1t, p->o_b1, p->H1, p->H1t, p->Z1);
    layer(p->H1, p->kh(), p->W2t, p->o_b2, p->H2, p->H2t, p->Z2);
}

// inference of the staged X into Y
void forward(g2g_mlp_s* p, int M, float* Y)
{
    hidden(p, M, false);
    GemmArgs a = operands(p->H2, p->kh(), p->W3t, p->kh(), M, p->n_out, p->kh());
    a.bias = p->w + p->o_b3;
    a.C = Y;
    a.ldc = p->n_out;
    product<kEpiBiasF32>(p, a);
}

// loss (p->loss[0]) and gradients (p->g), with their squared norm
// (p->loss[1]), of the staged X against the targets T (device)
void loss_and_grads(g2g_mlp_s* p, const float* T, int M)
{
    const int mt = g2g_mlp_s::pad8(M), H = p->H;
    hidden(p, M, true);
    // output layer: the loss's derivative straight from the product
    const float scale = static_cast<float>(1.0 / (static_cast<double>(M) * p->n_out));
    GemmArgs a = operands(p->H2, p->kh(), p->W3t, p->kh(), M, p->n_out, p->kh());
    a.bias = p->w + p->o_b3;
    a.T = T;
    a.ldc = p->n_out;
    a.scale = scale;
    a.H = p->dYb;
    a.ldh = p->kout();
    a.Ht = p->dYt;
    a.Mt = mt;
    a.colsum = p->cs3;
    a.sums = p->loss_sums;
    const size_t n_loss = product<kEpiMse>(p, a);
    size_t n_sums = 0;
    auto grad = [&](const __bf16* A, int rows, const __bf16* B, int cols, size_t off) {
        GemmArgs q = operands(A, mt, B, mt, rows, cols, mt);
        q.C = p->g + off;
        q.ldc = cols;
        q.sums = p->sums + n_sums;
        n_sums += product<kEpiGrad>(p, q);
    };
    auto back = [&](const __bf16* A, int ka, const __bf16* Wn, __bf16* Hh, __bf16* Ht, float* Z, float* cs) {
        GemmArgs q = operands(A, ka, Wn, ka, M, H, ka);
        q.H = Hh;
        q.ldh = p->kh();
        q.Ht = Ht;
        q.Mt = mt;
        q.Z = Z;
        q.ldz = H;
        q.colsum = cs;
        product<kEpiGeluBwd>(p, q);
    };
    grad(p->H2t, H, p->dYt, p->n_out, p->o_W3);
    back(p->dYb, p->kout(), p->W3n, p->dZ2b, p->dZ2t, p->Z2, p->cs2);
    grad(p->H1t, H, p->dZ2t, H, p->o_W2);
    back(p->dZ2b, p->kh(), p->W2n, nullptr, p->dZ1t, p->Z1, p->cs1);
    grad(p->Xt, p->n_in, p->dZ1t, H, p->o_W1);
    const BiasGradArgs b{{{static_cast<long long>(p->o_b1), static_cast<long long>(p->o_b2),
                           static_cast<long long>(p->o_b3)},
                          {H, H, p->n_out}},
                         {p->cs1, p->cs2, p->cs3},
                         (M + 31) / 32,
                         p->g,
                         p->sums + n_sums};
    const unsigned nb = blocks_for(2LL * H + p->n_out, 256);
    k_bias_grad<<<nb, 256, 0, p->stream>>>(b);
    n_sums += nb;
    k_finish<<<1, 1024, 0, p->stream>>>(p->loss_sums, static_cast<int>(n_loss), scale, p->sums,
                                        static_cast<int>(n_sums), p->loss, p->loss + 1);
    HIPCHK(hipGetLastError());
}

// the targets on the device: the caller's array, or its staged host copy
const float* stage_t(g2g_mlp_s* p, const float* T, int M, int on_device)
{
    if (on_device) return T;
    const size_t n = static_cast<size_t>(M) * p->n_out;
    HIPCHK(hipMemcpyAsync(p->T, T, n * sizeof(float), hipMemcpyHostToDevice, p->stream));
    HIPCHK(hipStreamSynchronize(p->stream));
    return p->T;
}

}  // namespace

namespace g2g {

// Warm-start voltages of rows [0, M) of a batch from its tiled Sbus (used by capi.cpp)
void mlp_warm_start_tiles(g2g_mlp_s* p, const double2* S_tiles, int M, int n, const unsigned char* d_mask, int n_mask,
                          double2* V_tiles, hipStream_t st)
{
    if (!p->kind) throw std::invalid_argument("the MLP has no bus types: call g2g_mlp_set_buses");
    if (p->n_bus != n) throw std::invalid_argument("the MLP's bus count differs from the batch's");
    if (p->n_in != 2 * n + n_mask) throw std::invalid_argument("the MLP's input width is not 2 n + mask");
    if (p->n_out != 2 * n) throw std::invalid_argument("the MLP's output width is not 2 n");
    if (!p->in_mu) throw std::invalid_argument("the MLP has no normalisation: call g2g_mlp_set_normalization");
    hipStream_t keep = p->stream;
    p->stream = st;
    p->workspace(M);
    const dim3 patches((n + kPatchBuses - 1) / kPatchBuses, (M + 63) / 64);
    k_features_tiles_t<<<patches, 256, 0, st>>>(S_tiles, M, n, p->in_mu, p->in_sigma, p->X, p->kin());
    if (n_mask > 0)
        k_mask_features<<<blocks_for(static_cast<long long>(M) * n_mask, 256), 256, 0, st>>>(d_mask, M, n, n_mask,
                                                                                            p->X, p->kin());
    HIPCHK(hipGetLastError());
    forward(p, M, p->Y);
    k_warm_v_tiles_t<<<patches, 256, 0, st>>>(p->Y, p->n_out, M, n, p->out_mu, p->out_sigma, p->vfix, p->kind,
                                              V_tiles);
    HIPCHK(hipGetLastError());
    p->stream = keep;
}

}  // namespace g2g

extern "C" {

int g2g_mlp_create(int32_t n_in, int32_t n_hidden, int32_t n_out, uint64_t seed, void* stream, g2g_mlp_t* out)
{
    return guarded([&] {
        if (!out) throw std::invalid_argument("null argument");
        if (n_in <= 0 || n_hidden <= 0 || n_out <= 0) throw std::invalid_argument("layer widths must be positive");
        auto p = std::make_unique<g2g_mlp_s>();
        p->n_in = n_in;
        p->H = n_hidden;
        p->n_out = n_out;
        p->stream = static_cast<hipStream_t>(stream);
        size_t o = 0;
        auto take = [&](size_t n) { const size_t at = o; o += (n + 63) / 64 * 64; return at; };
        p->o_W1 = take(static_cast<size_t>(n_in) * n_hidden);
        p->o_b1 = take(n_hidden);
        p->o_W2 = take(static_cast<size_t>(n_hidden) * n_hidden);
        p->o_b2 = take(n_hidden);
        p->o_W3 = take(static_cast<size_t>(n_hidden) * n_out);
        p->o_b3 = take(n_out);
        p->n_params = o;
        p->w = p->own.get<float>(o);
        p->m = p->own.get<float>(o);
        p->v = p->own.get<float>(o);
        p->g = p->own.get<float>(o);
        p->W1t = p->own.get<__bf16>(static_cast<size_t>(n_hidden) * p->kin());
        p->W2t = p->own.get<__bf16>(static_cast<size_t>(n_hidden) * p->kh());
        p->W3t = p->own.get<__bf16>(static_cast<size_t>(n_out) * p->kh());
        p->W2n = p->own.get<__bf16>(static_cast<size_t>(n_hidden) * p->kh());
        p->W3n = p->own.get<__bf16>(static_cast<size_t>(n_hidden) * p->kout());
        // Glorot-uniform weights, zero biases (seeded)
        std::vector<float> h(o, 0.0f);
        std::mt19937_64 rng(seed);
        auto fill = [&](size_t at, int fan_in, int fan_out) {
            const float a = std::sqrt(6.0f / static_cast<float>(fan_in + fan_out));
            std::uniform_real_distribution<float> u(-a, a);
            for (size_t i = 0; i < static_cast<size_t>(fan_in) * fan_out; ++i) h[at + i] = u(rng);
        };
        fill(p->o_W1, n_in, n_hidden);
        fill(p->o_W2, n_hidden, n_hidden);
        fill(p->o_W3, n_hidden, n_out);
        HIPCHK(hipMemcpy(p->w, h.data(), o * sizeof(float), hipMemcpyHostToDevice));
        HIPCHK(hipMemset(p->m, 0, o * sizeof(float)));
        HIPCHK(hipMemset(p->v, 0, o * sizeof(float)));
        // (the padding between the layers' gradients is never written; callers
        // that take the gradients copy it)
        HIPCHK(hipMemset(p->g, 0, o * sizeof(float)));
        p->refresh_weights(nullptr, nullptr);
        HIPCHK(hipDeviceSynchronize());
        *out = p.release();
    });
}

void g2g_mlp_destroy(g2g_mlp_t p)
{
    if (!p) return;
    (void)hipStreamSynchronize(p->stream);
    DeviceScratch::free_one(p->in_mu);
    DeviceScratch::free_one(p->in_sigma);
    DeviceScratch::free_one(p->out_mu);
    DeviceScratch::free_one(p->out_sigma);
    DeviceScratch::free_one(p->kind);
    DeviceScratch::free_one(p->vfix);
    delete p;
}

int64_t g2g_mlp_num_params(g2g_mlp_t p) { return p ? static_cast<int64_t>(p->n_params) : -1; }

int g2g_mlp_param_offsets(g2g_mlp_t p, int64_t* offsets)
{
    return guarded([&] {
        if (!p || !offsets) throw std::invalid_argument("null argument");
        const size_t o[6] = {p->o_W1, p->o_b1, p->o_W2, p->o_b2, p->o_W3, p->o_b3};
        for (int i = 0; i < 6; ++i) offsets[i] = static_cast<int64_t>(o[i]);
    });
}

int g2g_mlp_get_params(g2g_mlp_t p, float* out, int64_t capacity)
{
    return guarded([&] {
        if (!p || !out) throw std::invalid_argument("null argument");
        if (capacity < static_cast<int64_t>(p->n_params)) throw std::invalid_argument("output buffer too small");
        HIPCHK(hipStreamSynchronize(p->stream));
        HIPCHK(hipMemcpy(out, p->w, p->n_params * sizeof(float), hipMemcpyDeviceToHost));
    });
}

int g2g_mlp_set_params(g2g_mlp_t p, const float* in, int64_t n)
{
    return guarded([&] {
        if (!p || !in) throw std::invalid_argument("null argument");
        if (n != static_cast<int64_t>(p->n_params)) throw std::invalid_argument("parameter count mismatch");
        HIPCHK(hipStreamSynchronize(p->stream));
        HIPCHK(hipMemcpy(p->w, in, p->n_params * sizeof(float), hipMemcpyHostToDevice));
        p->refresh_weights(p->stream, nullptr);
        HIPCHK(hipStreamSynchronize(p->stream));
    });
}

int g2g_mlp_set_normalization(g2g_mlp_t p, const float* in_mu, const float* in_sigma, const float* out_mu,
                              const float* out_sigma)
{
    return guarded([&] {
        if (!p || !in_mu || !in_sigma || !out_mu || !out_sigma) throw std::invalid_argument("null argument");
        auto up = [&](float*& dst, const float* src, int n) {
            if (!dst) dst = dalloc<float>(static_cast<size_t>(n));
            HIPCHK(hipMemcpy(dst, src, static_cast<size_t>(n) * sizeof(float), hipMemcpyHostToDevice));
        };
        up(p->in_mu, in_mu, p->n_in);
        up(p->in_sigma, in_sigma, p->n_in);
        up(p->out_mu, out_mu, p->n_out);
        up(p->out_sigma, out_sigma, p->n_out);
    });
}

int g2g_mlp_set_buses(g2g_mlp_t p, const int32_t* kind, const double* vfix, int32_t n)
{
    return guarded([&] {
        if (!p || !kind || !vfix) throw std::invalid_argument("null argument");
        if (n <= 0) throw std::invalid_argument("n must be positive");
        DeviceScratch::free_one(p->kind);
        DeviceScratch::free_one(p->vfix);
        p->kind = dupload(std::vector<int>(kind, kind + n));
        p->vfix = dupload(std::vector<double>(vfix, vfix + n));
        p->n_bus = n;
    });
}

int g2g_mlp_forward(g2g_mlp_t p, const float* X, int32_t M, float* Y, int32_t on_device)
{
    return guarded([&] {
        if (!p || !X || !Y) throw std::invalid_argument("null argument");
        if (M <= 0) throw std::invalid_argument("M must be positive");
        p->workspace(M);
        stage_x(p, X, M, on_device, false);
        forward(p, M, on_device ? Y : p->Y);
        if (!on_device)
            HIPCHK(hipMemcpyAsync(Y, p->Y, static_cast<size_t>(M) * p->n_out * sizeof(float), hipMemcpyDeviceToHost,
                                  p->stream));
        HIPCHK(hipStreamSynchronize(p->stream));
    });
}

int g2g_mlp_loss_grad(g2g_mlp_t p, const float* X, const float* T, int32_t M, float* loss, float* grads,
                      int32_t on_device)
{
    return guarded([&] {
        if (!p || !X || !T) throw std::invalid_argument("null argument");
        if (M <= 0) throw std::invalid_argument("M must be positive");
        p->train_workspace(M);
        stage_x(p, X, M, on_device, true);
        loss_and_grads(p, stage_t(p, T, M, on_device), M);
        if (loss) HIPCHK(hipMemcpyAsync(loss, p->loss, sizeof(float), hipMemcpyDeviceToHost, p->stream));
        if (grads)
            HIPCHK(hipMemcpyAsync(grads, p->g, p->n_params * sizeof(float), hipMemcpyDeviceToHost, p->stream));
        HIPCHK(hipStreamSynchronize(p->stream));
    });
}

int g2g_mlp_train_step(g2g_mlp_t p, const float* X, const float* T, int32_t M, float lr, float* loss,
                       int32_t on_device)
{
    return guarded([&] {
        if (!p || !X || !T) throw std::invalid_argument("null argument");
        if (M <= 0) throw std::invalid_argument("M must be positive");
        p->train_workspace(M);
        stage_x(p, X, M, on_device, true);
        loss_and_grads(p, stage_t(p, T, M, on_device), M);
        ++p->step;
        const float b1 = 0.9f, b2 = 0.999f;
        const float c1 = 1.0f / (1.0f - std::pow(b1, static_cast<float>(p->step)));
        const float c2 = 1.0f / (1.0f - std::pow(b2, static_cast<float>(p->step)));
        const AdamArgs a{lr, b1, b2, 1e-8f, c1, c2, p->clip > 0.0f ? p->loss + 1 : nullptr, p->clip};
        p->refresh_weights(p->stream, &a);
        if (loss) {
            HIPCHK(hipMemcpyAsync(loss, p->loss, sizeof(float), hipMemcpyDeviceToHost, p->stream));
            HIPCHK(hipStreamSynchronize(p->stream));
        }
    });
}

int g2g_mlp_set_grad_clip(g2g_mlp_t p, float max_norm)
{
    return guarded([&] {
        if (!p) throw std::invalid_argument("null argument");
        if (!(max_norm >= 0.0f)) throw std::invalid_argument("max_norm must be >= 0 (0: off)");
        p->clip = max_norm;
    });
}

int g2g_gemm_bf16(int32_t trans_a, int32_t trans_b, int32_t M, int32_t N, int32_t K, const uint16_t* A, int64_t lda,
                  const uint16_t* B, int64_t ldb, float* C, int64_t ldc)
{
    return guarded([&] {
        if (!A || !B || !C) throw std::invalid_argument("null argument");
        if (M <= 0 || N <= 0 || K <= 0) throw std::invalid_argument("sizes must be positive");
        const size_t na = static_cast<size_t>(trans_a ? K : M) * static_cast<size_t>(lda);
        const size_t nb = static_cast<size_t>(trans_b ? N : K) * static_cast<size_t>(ldb);
        DeviceScratch s;
        __bf16* dA = s.get<__bf16>(na);
        __bf16* dB = s.get<__bf16>(nb);
        float* dC = s.get<float>(static_cast<size_t>(M) * ldc);
        HIPCHK(hipMemcpy(dA, A, na * 2, hipMemcpyHostToDevice));
        HIPCHK(hipMemcpy(dB, B, nb * 2, hipMemcpyHostToDevice));
        if (!trans_a && !trans_b) gemm<false, false>(nullptr, dA, lda, dB, ldb, M, N, K, dC, ldc);
        else if (!trans_a && trans_b && K % 8 == 0 && lda % 8 == 0 && ldb % 8 == 0)
        {
            GemmArgs a = operands(dA, lda, dB, ldb, M, N, K);
            a.C = dC;
            a.ldc = ldc;
            k_gemm_kc<kEpiF32><<<dim3((N + 127) / 128, (M + 127) / 128), 256>>>(a);
            HIPCHK(hipGetLastError());
        }
        else if (!trans_a && trans_b) gemm<false, true>(nullptr, dA, lda, dB, ldb, M, N, K, dC, ldc);
        else if (trans_a && !trans_b) gemm<true, false>(nullptr, dA, lda, dB, ldb, M, N, K, dC, ldc);
        else gemm<true, true>(nullptr, dA, lda, dB, ldb, M, N, K, dC, ldc);
        HIPCHK(hipDeviceSynchronize());
        HIPCHK(hipMemcpy(C, dC, static_cast<size_t>(M) * ldc * sizeof(float), hipMemcpyDeviceToHost));
    });
}

}  // extern "C"
