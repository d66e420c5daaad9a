// One training step of the surrogate network (nfeat -> 256 -> 256 -> 256 -> 8,
// GELU) in three launches: forward, loss and the chain of activation
// gradients for a block of rows; the weight gradients; Adam.  No reference
// counterpart.  The same arithmetic as tt_gemm_bf16 / tt_gelu_backward /
// tt_surrogate_loss / tt_adam called layer by layer (bf16 operands, fp32
// accumulation over k in steps of 32, fp32 pre-activations and gradients, the
// same roundings to bf16, the same partial sums of a gradient); those partial
// sums are added in order, where the atomic adds there take any.
//
// What bounds a step: at 8192 rows its 7.1 GFLOP take 6 us of the matrix cores
// and its bytes less; called layer by layer it was 45 launches of 1 to 30 us,
// 433 us, of which the products spent most on atomic adds of weight gradients
// and 130 us went to column sums by 32 waves.  In three launches it is 62 us:
// 39 for the rows, 18 for the weight gradients, 5 for Adam, each bound by the
// latency of its own chain of dependent loads and products.
#include "gelu.h"
#include "tt_internal.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int kH = 256;        // hidden width
constexpr int kOut = 8;        // outputs
constexpr int kLd = kH + 8;    // LDS row of activations (bf16): 16-byte rows, spread over the banks
constexpr int kXLd = 64 + 8;   // LDS row of input features
constexpr int kChunk = 32;     // rows per K step of the weight gradients

struct LossDev {
    const float *T;
    int64_t ldt;
    int n_reg, n_err;
    float w[8];
    int lo[4], hi[4];
    float tau;
    double *sums;
};

struct StepArgs {
    const __bf16 *X;  // [.][ldx]
    int64_t ldx;
    const int64_t *rows;  // the batch's rows of X and T
    int n, nfeat;
    const __bf16 *w[4];   // [out][in]
    const __bf16 *wt[4];  // [in][out], layers 1..3
    const float *b[4];
    LossDev loss;
    // operands of the weight gradients, [chunk of 32 rows][feature][row]
    __bf16 *act[4];   // layer l's input, kH features (64 for l = 0)
    __bf16 *grad[4];  // layer l's pre-activation gradient, kH features (16 for l = 3)
};

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ bf16x8 zero8() {
    return bf16x8{(__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f};
}

// A wave owns 32 of a layer's 256 features: two 16-feature tiles of M H^T for
// the block's 16 T rows, M [256][ldm] (row = feature) and the activations in
// LDS as [row][ld].  K = 32 KC; columns at or beyond kvalid (a multiple of 8)
// count as zero.  The weight fragments are loaded apart from the products, a
// layer ahead.
constexpr int kWaves = 8, kThreads = 64 * kWaves;

template <int KC>
struct Frags {
    bf16x8 a[2][KC];
    __device__ __forceinline__ void load(const __bf16 *M, int ldm, int kvalid) {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
            for (int c = 0; c < KC; ++c) {
                const int k = 32 * c + 8 * g;
                a[nt][c] = k < kvalid ? *reinterpret_cast<const bf16x8 *>(M + (32 * wave + 16 * nt + r) * ldm + k) : zero8();
            }
    }
    template <int T>
    __device__ __forceinline__ void product(const __bf16 *in, int ld, int kvalid, f32x4 (&acc)[2][T]) const {
        const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
            for (int t = 0; t < T; ++t) acc[nt][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < KC; ++c) {
            bf16x8 x[T];
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const int k = 32 * c + 8 * g;
                x[t] = k < kvalid ? *reinterpret_cast<const bf16x8 *>(in + (16 * t + r) * ld + k) : zero8();
            }
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                for (int t = 0; t < T; ++t) acc[nt][t] = mfma(a[nt][c], x[t], acc[nt][t]);
        }
    }
};

// the block's activations [16 T rows][256] from LDS to chunk order in memory:
// half the rows of one feature per thread, its rows consecutive
template <int T>
__device__ __forceinline__ void put_chunks(const __bf16 *lds, int ld, int nf, int row0, __bf16 *out) {
    const int f = threadIdx.x & 255, half = threadIdx.x >> 8;
    if (f >= nf) return;
    __bf16 *o = out + ((int64_t)(row0 / kChunk) * nf + f) * kChunk + row0 % kChunk;
#pragma unroll
    for (int p = 0; p < T; ++p) {
        const int q = half * T + p;
        bf16x8 v;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = lds[(8 * q + j) * ld + f];
        *reinterpret_cast<bf16x8 *>(o + 8 * q) = v;
    }
}

// Forward, loss and activation gradients of 16 T rows.  A wave owns the same 32
// of the 256 features in every layer, forward and backward, so a layer's
// pre-activations stay in its registers until the backward pass needs them:
// nothing but the operands of the weight gradients is written.  Activations
// pass between the waves through two LDS tiles.  0.55 MB of weights per block
// come from L2; seven products and as many barriers follow one another, so the
// time is their latency, and each product's fragments are loaded while the one
// before is finished.  T = 2 (256 blocks at 8192 rows, one per CU) or 1 below
// 8192 rows, where T = 2 would leave CUs idle.  The rows go to the XCDs in
// contiguous eighths, the splits of the weight gradients likewise, so those
// find their operands in their own L2.
template <int T>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void train_rows_kernel(StepArgs a) {
    constexpr int R = 16 * T;
    __shared__ __attribute__((aligned(16))) __bf16 xs[R * kXLd], h0[R * kLd], h1[R * kLd], dys[R * 16];
    __shared__ float ys[R * kOut];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const int row0 = tt::xcd_block((int)blockIdx.x, (int)gridDim.x) * R;
    Frags<2> wx;
    Frags<8> wa, wb;
    Frags<1> wo;
    wx.load(a.w[0], a.nfeat, a.nfeat);
    // wave 0's lanes take a row each for the loss: its targets, asked for early
    float target[8];
    const bool has_row = wave == 0 && lane < R && row0 + lane < a.n;
#pragma unroll
    for (int j = 0; j < 8; ++j)
        target[j] = has_row && j < a.loss.n_reg ? a.loss.T[a.rows[row0 + lane] * a.loss.ldt + j] : 0.f;
    for (int i = threadIdx.x; i < R * 8; i += kThreads) {
        const int row = i >> 3, k = (i & 7) * 8;
        bf16x8 v = zero8();
        if (row0 + row < a.n && k < a.nfeat) v = *reinterpret_cast<const bf16x8 *>(a.X + a.rows[row0 + row] * a.ldx + k);
        *reinterpret_cast<bf16x8 *>(&xs[row * kXLd + k]) = v;
    }
    for (int i = threadIdx.x; i < R * 16; i += kThreads) dys[i] = (__bf16)0.f;
    tt::lds_barrier();
    put_chunks<T>(xs, kXLd, 64, row0, a.act[0]);
    f32x4 z[3][2][T], acc[2][T];
    __bf16 *tile[2] = {h0, h1};
    // a layer's pre-activations -> its activations, in LDS and for the weight gradients
    auto activate = [&](int l, __bf16 *out) __attribute__((always_inline)) {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            const int f = 32 * wave + 16 * nt + 4 * g;
            const float4 bb = *reinterpret_cast<const float4 *>(a.b[l] + f);
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const f32x4 v = {acc[nt][t][0] + bb.x, acc[nt][t][1] + bb.y, acc[nt][t][2] + bb.z, acc[nt][t][3] + bb.w};
                z[l][nt][t] = v;
                bf16x4 h;
#pragma unroll
                for (int i = 0; i < 4; ++i) h[i] = (__bf16)tt::gelu_f(v[i]);
                *reinterpret_cast<bf16x4 *>(&out[(16 * t + r) * kLd + f]) = h;
            }
        }
        tt::lds_barrier();
        put_chunks<T>(out, kLd, kH, row0, a.act[l + 1]);
    };
    wa.load(a.w[1], kH, kH);
    wx.product<T>(xs, kXLd, a.nfeat, acc);
    wb.load(a.w[2], kH, kH);
    activate(0, tile[0]);
    wa.product<T>(tile[0], kLd, kH, acc);
    wo.load(a.wt[3], kOut, kOut);
    activate(1, tile[1]);
    wb.product<T>(tile[1], kLd, kH, acc);
    wa.load(a.wt[2], kH, kH);
    activate(2, tile[0]);
    // the outputs: wave t takes row tile t
    if (wave < T) {
        bf16x8 w[8];
#pragma unroll
        for (int c = 0; c < 8; ++c)
            w[c] = r < kOut ? *reinterpret_cast<const bf16x8 *>(a.w[3] + r * kH + 32 * c + 8 * g) : zero8();
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 8; ++c)
            o = mfma(w[c], *reinterpret_cast<const bf16x8 *>(&tile[0][(16 * wave + r) * kLd + 32 * c + 8 * g]), o);
        if (g < 2)
#pragma unroll
            for (int i = 0; i < 4; ++i) ys[(16 * wave + r) * kOut + 4 * g + i] = o[i] + a.b[3][4 * g + i];
    }
    tt::lds_barrier();
    // loss and its gradient (tt_surrogate_loss)
    double s2 = 0.0, s1 = 0.0;
    if (has_row) {
        const LossDev &q = a.loss;
        const float *y = ys + lane * kOut;
        __bf16 *d = dys + lane * 16;
        const float inv = 1.0f / (float)a.n;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (j >= q.n_reg) break;
            const float e = y[j] - target[j];
            s2 += (double)(q.w[j] * e * e);
            d[j] = (__bf16)(2.0f * q.w[j] * e * inv);
        }
        for (int h = 0; h < q.n_err; ++h) {
            float far = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (j >= q.lo[h] && j < q.hi[h]) far = fmaxf(far, fabsf(target[j] - y[j]));
            const float e = y[q.n_reg + h] - far;
            s1 += (double)(e > 0.f ? (1.0f - q.tau) * e : -q.tau * e);
            d[q.n_reg + h] = (__bf16)((e > 0.f ? 1.0f - q.tau : (e < 0.f ? -q.tau : 0.0f)) * inv);
        }
    }
    tt::lds_barrier();
    put_chunks<T>(dys, 16, 16, row0, a.grad[3]);
    // gradient of a layer's pre-activations from that of its activations
    auto back = [&](int l, __bf16 *out) __attribute__((always_inline)) {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
            for (int t = 0; t < T; ++t) {
                bf16x4 d;
#pragma unroll
                for (int i = 0; i < 4; ++i) d[i] = (__bf16)(acc[nt][t][i] * tt::gelu_grad(z[l][nt][t][i]));
                *reinterpret_cast<bf16x4 *>(&out[(16 * t + r) * kLd + 32 * wave + 16 * nt + 4 * g]) = d;
            }
        tt::lds_barrier();
        put_chunks<T>(out, kLd, kH, row0, a.grad[l]);
    };
    wo.product<T>(dys, 16, kOut, acc);
    wb.load(a.wt[1], kH, kH);
    back(2, tile[1]);
    wa.product<T>(tile[1], kLd, kH, acc);
    back(1, tile[0]);
    wb.product<T>(tile[0], kLd, kH, acc);
    back(0, tile[1]);
    if (wave == 0) {
        for (int off = 32; off > 0; off >>= 1) {
            s2 += __shfl_down(s2, off, 64);
            s1 += __shfl_down(s1, off, 64);
        }
        if (lane == 0) {
            atomicAdd(&a.loss.sums[0], s2);
            atomicAdd(&a.loss.sums[1], s1);
        }
    }
}

// Weight gradients dW[out][in] = sum over rows dZ[row][out] A[row][in] and bias
// gradients, all layers in one launch.  A block takes one 64 x 64 tile of one
// layer and one of the splits of the rows, each wave a 32 x 32 quarter of the
// tile.  In chunk order both operands' fragments are contiguous 1 KB loads, so
// there is no LDS staging, and the next chunk's are in flight during this
// one's products.  A split's rows are added in order and its partial tile is
// written for Adam to add: the partial sums of tt_gemm_bf16's split K in a
// fixed order, without its atomic adds into dW, which took most of that
// kernel's time.  The first blocks add up columns of dZ for the bias
// gradients as tt_bias_grad does, kBiasRows rows in order per thread.
constexpr int kTiles = 4 + 16 + 16 + 4;  // layers 0..3
constexpr int kPart = 64 * 64;           // a partial tile
constexpr int kBiasCols = 3 * kH + kOut;
constexpr int kBiasRows = 256;

struct GradArgs {
    const __bf16 *act[4], *grad[4];
    int chunks, per_split;  // chunks of 32 rows in all, in a split
    float *part;            // [splits][kTiles][kPart]
    float *bias;            // [groups of kBiasRows rows][kBiasCols]
};

__device__ __forceinline__ void bias_grad(const GradArgs &a, int group, int col) {
    if (col >= kBiasCols) return;
    const int l = col < 3 * kH ? col / kH : 3, fg = l == 3 ? 16 : kH;
    const __bf16 *p = a.grad[l] + (int64_t)(col - l * kH) * kChunk;
    const int c0 = group * (kBiasRows / kChunk), c1 = min(a.chunks, c0 + kBiasRows / kChunk);
    constexpr int NC = kBiasRows / kChunk, NQ = kChunk / 8;
    bf16x8 v[NC][NQ];  // all loads in flight together
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int q = 0; q < NQ; ++q)
            v[c][q] = c0 + c < c1 ? *reinterpret_cast<const bf16x8 *>(p + (int64_t)(c0 + c) * fg * kChunk + 8 * q) : zero8();
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int j = 0; j < 8; ++j) s += (float)v[c][q][j];
    a.bias[group * kBiasCols + col] = s;
}

__global__ __launch_bounds__(256) void weight_grad_kernel(GradArgs a, int splits, int groups) {
    constexpr int per = (kBiasCols + 255) / 256;
    if ((int)blockIdx.x < groups * per) {  // bias gradients, per blocks a group
        bias_grad(a, blockIdx.x / per, blockIdx.x % per * 256 + threadIdx.x);
        return;
    }
    // splits vary fastest: with eight of them, one per XCD
    const int id = (int)blockIdx.x - groups * per, split = id % splits, tile = id / splits;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    int l, ot, it;
    if (tile < 4) {
        l = 0, ot = tile, it = 0;
    } else if (tile < 36) {
        l = 1 + (tile - 4) / 16, ot = (tile - 4) % 16 / 4, it = (tile - 4) % 4;
    } else {
        l = 3, ot = 0, it = tile - 36;
    }
    const int fa = l == 0 ? 64 : kH, fg = l == 3 ? 16 : kH;  // features per chunk
    const int o0 = 32 * (wave >> 1), i0 = 32 * (wave & 1);   // this wave's quarter
    const int nto = l == 3 ? (o0 ? 0 : 1) : 2;               // its 16-row tiles of outputs
    if (nto == 0) return;
    const int c0 = split * a.per_split, c1 = min(a.chunks, c0 + a.per_split);
    f32x4 acc[2][2];
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int m = 0; m < 2; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    const __bf16 *pg = a.grad[l] + (int64_t)(64 * ot + o0 + r) * kChunk + 8 * g;
    const __bf16 *pa = a.act[l] + (int64_t)(64 * it + i0 + r) * kChunk + 8 * g;
    constexpr int A = 6;  // chunks in flight
    bf16x8 x[A][2], y[A][2];
    auto fetch = [&](int c, bf16x8 (&u)[2], bf16x8 (&v)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            u[n] = n < nto ? *reinterpret_cast<const bf16x8 *>(pg + ((int64_t)c * fg + 16 * n) * kChunk) : zero8();
            v[n] = *reinterpret_cast<const bf16x8 *>(pa + ((int64_t)c * fa + 16 * n) * kChunk);
        }
    };
#pragma unroll
    for (int j = 0; j < A; ++j)
        if (c0 + j < c1) fetch(c0 + j, x[j], y[j]);
    for (int c = c0; c < c1; c += A)
#pragma unroll
        for (int j = 0; j < A; ++j) {
            if (c + j >= c1) break;
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int m = 0; m < 2; ++m) acc[n][m] = mfma(x[j][n], y[j][m], acc[n][m]);
            if (c + j + A < c1) fetch(c + j + A, x[j], y[j]);
        }
    float *out = a.part + ((int64_t)split * kTiles + tile) * kPart;
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) out[(o0 + 16 * n + 4 * g + i) * 64 + i0 + 16 * m + r] = acc[n][m][i];
}

// Adam (tt_adam) over all weights and biases, gradients added up from their
// partial tiles; refreshes the bf16 copies and their transposes.
struct AdamArgs {
    float *w[4], *b[4], *dw[4], *db[4], *mw[4], *vw[4], *mb[4], *vb[4];
    __bf16 *wb[4], *wt[4];
    const float *part, *bias;
    int splits, groups, nfeat;
    float lr, b1, b2, eps, c1, c2, wd;
};

__global__ __launch_bounds__(256) void step_adam_kernel(AdamArgs a) {
    int i = blockIdx.x * 256 + threadIdx.x;
    const int nw[4] = {kH * a.nfeat, kH * kH, kH * kH, kOut * kH};
    int l = 0, o, k;
    bool bias = false;
    while (l < 4 && i >= nw[l]) i -= nw[l++];
    if (l == 4) {  // biases
        bias = true;
        l = i < 3 * kH ? i / kH : 3;
        i -= l * kH;
        if (l == 3 && i >= kOut) return;
        o = i, k = 0;
    } else {
        const int fin = l == 0 ? a.nfeat : kH;
        o = i / fin, k = i - o * fin;
    }
    float gsum = 0.f;
    if (bias) {
#pragma unroll 8
        for (int q = 0; q < a.groups; ++q) gsum += a.bias[q * kBiasCols + l * kH + o];
    } else {
        const int tile = l == 0 ? o / 64 : l == 3 ? 36 + k / 64 : 4 + 16 * (l - 1) + 4 * (o / 64) + k / 64;
        const float *p = a.part + (int64_t)tile * kPart + (o % 64) * 64 + k % 64;
#pragma unroll 8
        for (int q = 0; q < a.splits; ++q) gsum += p[(int64_t)q * kTiles * kPart];
    }
    float *w = bias ? a.b[l] : a.w[l], *m = bias ? a.mb[l] : a.mw[l], *v = bias ? a.vb[l] : a.vw[l];
    (bias ? a.db[l] : a.dw[l])[i] = gsum;
    const float gi = gsum + (bias ? 0.f : a.wd) * w[i];
    const float mi = a.b1 * m[i] + (1.0f - a.b1) * gi;
    const float vi = a.b2 * v[i] + (1.0f - a.b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float wi = w[i] - a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
    w[i] = wi;
    if (!bias) {
        a.wb[l][i] = (__bf16)wi;
        if (l > 0) a.wt[l][k * (l == 3 ? kOut : kH) + o] = (__bf16)wi;
    }
}

int chunks_of(int batch) { return (int)tt::ceil_div(batch, kChunk); }
// rows per split of the weight gradients: those of MLP.backward's products
int split_rows(int batch) { return batch >= 2048 ? 1024 : chunks_of(batch) * kChunk; }
int splits_of(int batch) { return (int)tt::ceil_div(batch, split_rows(batch)); }
int groups_of(int batch) { return (int)tt::ceil_div(batch, kBiasRows); }

struct Layout {
    size_t act[4], grad[4], part, bias, total;
};
Layout layout_of(int batch) {
    Layout L;
    size_t at = 0;
    auto take = [&](size_t bytes) {
        const size_t p = at;
        at += (bytes + 255) / 256 * 256;
        return p;
    };
    const size_t rows = (size_t)chunks_of(batch) * kChunk;
    for (int l = 0; l < 4; ++l) {
        L.act[l] = take(rows * (l == 0 ? 64 : kH) * sizeof(__bf16));
        L.grad[l] = take(rows * (l == 3 ? 16 : kH) * sizeof(__bf16));
    }
    L.part = take((size_t)splits_of(batch) * kTiles * kPart * sizeof(float));
    L.bias = take((size_t)groups_of(batch) * kBiasCols * sizeof(float));
    L.total = at;
    return L;
}

}  // namespace

extern "C" int tt_mlp_train_workspace_bytes(int32_t batch, size_t *bytes) {
    TT_REQUIRE(bytes && batch >= 1 && batch <= (1 << 24), "tt_mlp_train_workspace_bytes: need 1 <= batch <= 2^24");
    *bytes = layout_of(batch).total;
    return TT_OK;
}

extern "C" int tt_mlp_train_step(const tt_mlp_train *s, void *stream) {
    TT_REQUIRE(s, "tt_mlp_train_step: null arguments");
    TT_REQUIRE(s->batch >= 1 && s->batch <= (1 << 24), "tt_mlp_train_step: need 1 <= batch <= 2^24");
    TT_REQUIRE(s->nfeat >= 8 && s->nfeat <= 64 && s->nfeat % 8 == 0,
               "tt_mlp_train_step: nfeat must be a multiple of 8 in [8, 64]");
    TT_REQUIRE(s->X && s->T && s->rows && s->loss_out && s->workspace, "tt_mlp_train_step: null pointer");
    TT_REQUIRE(s->ldx >= s->nfeat && s->ldx % 8 == 0 && ((uintptr_t)s->X & 15) == 0,
               "tt_mlp_train_step: rows of X must be 16-byte aligned");
    TT_REQUIRE(s->n_reg >= 1 && s->n_err >= 0 && s->n_err <= 4 && s->n_reg + s->n_err <= kOut && s->ldt >= s->n_reg,
               "tt_mlp_train_step: bad column counts");
    TT_REQUIRE(s->tau > 0.0 && s->tau < 1.0, "tt_mlp_train_step: tau must be in (0, 1)");
    TT_REQUIRE(s->step >= 1, "tt_mlp_train_step: step must be >= 1");
    const Layout L = layout_of(s->batch);
    TT_REQUIRE(s->workspace_bytes >= L.total && ((uintptr_t)s->workspace & 15) == 0,
               "tt_mlp_train_step: workspace of %zu bytes < %zu needed, or not 16-byte aligned", s->workspace_bytes,
               L.total);
    StepArgs a{};
    GradArgs g{};
    AdamArgs d{};
    char *ws = static_cast<char *>(s->workspace);
    for (int l = 0; l < 4; ++l) {
        const tt_mlp_layer &y = s->layer[l];
        TT_REQUIRE(y.w && y.b && y.w_bf16 && y.dw && y.db && y.mw && y.vw && y.mb && y.vb && (l == 0 || y.wt_bf16),
                   "tt_mlp_train_step: layer %d: null pointer", l);
        TT_REQUIRE((((uintptr_t)y.w_bf16 | (uintptr_t)y.wt_bf16 | (uintptr_t)y.b) & 15) == 0,
                   "tt_mlp_train_step: layer %d: weights and biases must be 16-byte aligned", l);
        a.w[l] = static_cast<const __bf16 *>(y.w_bf16);
        a.wt[l] = static_cast<const __bf16 *>(y.wt_bf16);
        a.b[l] = y.b;
        a.act[l] = reinterpret_cast<__bf16 *>(ws + L.act[l]);
        a.grad[l] = reinterpret_cast<__bf16 *>(ws + L.grad[l]);
        g.act[l] = a.act[l];
        g.grad[l] = a.grad[l];
        d.w[l] = y.w;
        d.b[l] = y.b;
        d.dw[l] = y.dw;
        d.db[l] = y.db;
        d.mw[l] = y.mw;
        d.vw[l] = y.vw;
        d.mb[l] = y.mb;
        d.vb[l] = y.vb;
        d.wb[l] = static_cast<__bf16 *>(y.w_bf16);
        d.wt[l] = static_cast<__bf16 *>(y.wt_bf16);
    }
    a.X = static_cast<const __bf16 *>(s->X);
    a.ldx = s->ldx;
    a.rows = s->rows;
    a.n = s->batch;
    a.nfeat = s->nfeat;
    a.loss.T = s->T;
    a.loss.ldt = s->ldt;
    a.loss.n_reg = s->n_reg;
    a.loss.n_err = s->n_err;
    for (int j = 0; j < s->n_reg; ++j) a.loss.w[j] = s->w_reg[j];
    for (int h = 0; h < s->n_err; ++h) {
        TT_REQUIRE(s->err_lo[h] >= 0 && s->err_hi[h] <= s->n_reg && s->err_lo[h] < s->err_hi[h],
                   "tt_mlp_train_step: bad error-head column range");
        a.loss.lo[h] = s->err_lo[h];
        a.loss.hi[h] = s->err_hi[h];
    }
    a.loss.tau = (float)s->tau;
    a.loss.sums = s->loss_out;
    hipStream_t st = tt::as_stream(stream);
    const int rows = chunks_of(s->batch) * kChunk;  // rows beyond the batch are zeros
    if (s->batch >= 8192)
        hipLaunchKernelGGL((train_rows_kernel<2>), dim3((unsigned)(rows / 32)), dim3(kThreads), 0, st, a);
    else
        hipLaunchKernelGGL((train_rows_kernel<1>), dim3((unsigned)(rows / 16)), dim3(kThreads), 0, st, a);
    TT_LAUNCH_CHECK("tt_mlp_train_step rows launch");
    g.chunks = rows / kChunk;
    g.per_split = split_rows(s->batch) / kChunk;
    g.part = reinterpret_cast<float *>(ws + L.part);
    g.bias = reinterpret_cast<float *>(ws + L.bias);
    const int splits = splits_of(s->batch), groups = groups_of(s->batch);
    const int64_t blocks = (int64_t)kTiles * splits + (int64_t)groups * tt::ceil_div(kBiasCols, 256);
    hipLaunchKernelGGL(weight_grad_kernel, dim3((unsigned)blocks), dim3(256), 0, st, g, splits, groups);
    TT_LAUNCH_CHECK("tt_mlp_train_step weight gradient launch");
    d.part = g.part;
    d.bias = g.bias;
    d.splits = splits;
    d.groups = groups;
    d.nfeat = s->nfeat;
    d.lr = (float)s->lr;
    d.b1 = (float)s->b1;
    d.b2 = (float)s->b2;
    d.eps = (float)s->eps;
    d.c1 = (float)(1.0 - pow(s->b1, (double)s->step));
    d.c2 = (float)(1.0 - pow(s->b2, (double)s->step));
    d.wd = (float)s->weight_decay;
    const int params = kH * s->nfeat + 2 * kH * kH + kOut * kH + 3 * kH + kOut;
    hipLaunchKernelGGL(step_adam_kernel, dim3((unsigned)tt::ceil_div(params, 256)), dim3(256), 0, st, d);
    TT_LAUNCH_CHECK("tt_mlp_train_step Adam launch");
    return TT_OK;
}
