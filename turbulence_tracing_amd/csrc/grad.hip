// Gradient stencil: the work of ElectronCube.calc_dndr
// (particle_tracking/particle_tracker.py:220-241) as one HBM-bound pass.
//
// For each node: ne/nc = alpha + beta f, clipped at ne_max (PT:230-231);
// -0.5 d(ne/nc)/dx_i by np.gradient's rule (central interior, one-sided
// first-order edges; PT:235-237); the result is written as one float4 per
// node {Gx, Gy, Gz, Phi} in the x-fastest/z-slowest layout the tracer reads:
//   G   = -0.5 dz grad(ne/nc)          (velocity change per z-cell)
//   Phi = k0 dz (sqrt(1 - ne/nc) - 1)  (phase per z-cell)
// Algorithmic traffic: sizeof(T) read + 16 B written per node.
#include <algorithm>

#include "tt_internal.h"

namespace {

template <typename T>
struct GradArgs {
    const T *f;
    int64_t sx, sy, sz;
    int nx, ny, nz;
    T beta, clipv;  // s = min(beta f, clipv); ne/nc = alpha + s
    double alpha;
    T cx, cy, cz;   // -0.5 dz / (2 d_i): scale of a central difference
    float phase_scale;  // k0 dz
    const double *sumsq; // optional: beta /= sqrt(*sumsq / count) (unit-RMS normalisation)
    double count;
    int run;            // planes per block along the march axis
    float4 *out;
};

// one-dimensional np.gradient at index i of n given the stencil values
template <typename T>
__device__ __forceinline__ T grad1(T sm, T s0, T sp, int i, int n, T c) {
    if (i == 0) return (sp - s0) * (c + c);
    if (i == n - 1) return (s0 - sm) * (c + c);
    return (sp - sm) * c;
}

// the node of stencil value s and gradient (gx, gy, gz), streamed past the caches
typedef float f32x4 __attribute__((ext_vector_type(4)));
template <typename T>
__device__ __forceinline__ void write_node(const GradArgs<T> &a, int ix, int iy, int iz, T s, T gx, T gy, T gz) {
    const double r = a.alpha + (double)s;
    const double q = 1.0 - r;
    // n - 1 = -r / (1 + sqrt(1 - r)), evaluated without cancellation
    const double eta = q > 0.0 ? -r / (1.0 + sqrt(q)) : -1.0;
    const f32x4 v = {(float)gx, (float)gy, (float)gz, (float)(eta * (double)a.phase_scale)};
    __builtin_nontemporal_store(v, reinterpret_cast<f32x4 *>(a.out + ((int64_t)iz * a.ny + iy) * a.nx + ix));
}

// One pass bound by HBM.  A block owns a tile of the plane of x and a second
// axis b (z if the input is contiguous along z, else y) and marches along the
// third axis c.  Each plane of the tile, with a halo of one node, is read once
// with the lanes along the input's contiguous axis and goes through LDS, where
// it turns to the output's x-fastest order; the neighbours in x and b come from
// LDS, those along c from registers.  Three buffers, so one barrier a plane (the
// buffer written was last read before the previous one), and the next plane's
// loads stay in flight across it.  The output, streamed past the caches, is
// four fifths of the bytes (fp32 input).
// Measured: 512^3 fp32 x-fastest 527 us (5.1 TB/s; 915 as a column walk that
// met its x and y neighbours in L1), 1024^3 3.93 ms (7.28), 201^3 fp64
// z-fastest 56 us (490 with strided lanes), 512^3 fp64 z-fastest 0.73 ms
// (7.13).  With eta left out 516 us: the fp64 root and quotient are hidden.
// Tiles of 64 x 16 where the lanes run along x (32 x 32: 552 us); 32 x 32 where
// they run along b, so both axes move at least 128 bytes at a time.

template <typename T, int TX, bool BZ, bool FASTX>
__global__ __launch_bounds__(256) void grad_kernel(GradArgs<T> a) {
    constexpr int TB = 1024 / TX, HX = TX + 2, HB = TB + 2, N = HX * HB, P = FASTX ? HX : HX | 1;
    constexpr int kLoads = (N + 255) / 256, kRows = 256 / TX, kOwn = TB / kRows;
    __shared__ T lds[3][HB * P];
    const int nb = BZ ? a.nz : a.ny, nc = BZ ? a.ny : a.nz;
    const int64_t sb = BZ ? a.sz : a.sy, sc = BZ ? a.sy : a.sz;
    const int x0 = (int)blockIdx.x * TX, b0 = (int)blockIdx.y * TB, c0 = (int)blockIdx.z * a.run;
    const int c1 = min(c0 + a.run, nc);
    // this thread's elements of a plane, halo included; coordinates beyond the
    // grid are clamped (grad1 leaves those values out)
    const T *src[kLoads];
    int dst[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int e = min((int)threadIdx.x + 256 * i, N - 1);
        const int ex = FASTX ? e % HX : e / HB, eb = FASTX ? e / HX : e % HB;
        const int gx = min(max(x0 + ex - 1, 0), a.nx - 1), gb = min(max(b0 + eb - 1, 0), nb - 1);
        src[i] = a.f + gx * a.sx + gb * sb;
        dst[i] = eb * P + ex;
    }
    T in[kLoads], in0[kLoads], in1[kLoads];
    const auto fetch = [&](T *v, int c) {
        const int64_t o = min(max(c, 0), nc - 1) * sc;
#pragma unroll
        for (int i = 0; i < kLoads; ++i) v[i] = src[i][o];
    };
    fetch(in0, c0 - 1);
    fetch(in1, c0);
    fetch(in, c0 + 1);
    T beta = a.beta;
    if (a.sumsq) beta = (T)((double)beta / sqrt(*a.sumsq / a.count));
    const auto stage = [&](const T *v, T *l) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const T s = v[i] * beta;
            if ((i + 1) * 256 <= N || (int)threadIdx.x + 256 * i < N) l[dst[i]] = s < a.clipv ? s : a.clipv;
        }
    };
    const int tx = threadIdx.x % TX, tb = threadIdx.x / TX;
    const int ix = x0 + tx;
    const int own = (tb + 1) * P + tx + 1;
    T cm[kOwn], s0[kOwn];
    stage(in0, lds[2]);
    stage(in1, lds[0]);
    tt::lds_barrier();
#pragma unroll
    for (int j = 0; j < kOwn; ++j) {
        cm[j] = lds[2][own + j * kRows * P];
        s0[j] = lds[0][own + j * kRows * P];
    }
    int cur = 0;
    for (int c = c0; c < c1; ++c) {
        // the plane staged three steps ago was last read before the barrier of the step before
        const int nxt = cur == 2 ? 0 : cur + 1;
        stage(in, lds[nxt]);
        fetch(in, c + 2);
        tt::lds_barrier();
        const T *l = lds[cur] + own, *ln = lds[nxt] + own;
#pragma unroll
        for (int j = 0; j < kOwn; ++j) {
            const int o = j * kRows * P;
            const int ib = b0 + tb + j * kRows;
            const T cp = ln[o];
            const T s = s0[j];
            const T gx = grad1(l[o - 1], s, l[o + 1], ix, a.nx, a.cx);
            const T gb = grad1(l[o - P], s, l[o + P], ib, nb, BZ ? a.cz : a.cy);
            const T gc = grad1(cm[j], s, cp, c, nc, BZ ? a.cy : a.cz);
            if (ix < a.nx && ib < nb) write_node(a, ix, BZ ? c : ib, BZ ? ib : c, s, gx, BZ ? gc : gb, BZ ? gb : gc);
            cm[j] = s;
            s0[j] = cp;
        }
        cur = nxt;
    }
}

// Grids of a few planes along b: those tiles would be mostly empty.  A thread walks
// one (x, y) column, carrying the z neighbours in registers and meeting those in x
// and y, which its block's 64 x 4 columns read together, in L1.
template <typename T>
__global__ __launch_bounds__(256) void grad_columns_kernel(GradArgs<T> a) {
    const int ix = (int)blockIdx.x * 64 + threadIdx.x % 64, iy = (int)blockIdx.y * 4 + threadIdx.x / 64;
    if (ix >= a.nx || iy >= a.ny) return;
    const int z0 = (int)blockIdx.z * a.run, z1 = min(z0 + a.run, a.nz);
    T beta = a.beta;
    if (a.sumsq) beta = (T)((double)beta / sqrt(*a.sumsq / a.count));
    const auto at = [&](int x, int y, int z) {
        const T v = a.f[x * a.sx + y * a.sy + z * a.sz] * beta;
        return v < a.clipv ? v : a.clipv;
    };
    T zm = z0 > 0 ? at(ix, iy, z0 - 1) : (T)0;
    T s0 = at(ix, iy, z0);
    for (int iz = z0; iz < z1; ++iz) {
        __builtin_amdgcn_s_setprio(1);  // the plane's loads leave before other waves' arithmetic
        const T zp = iz < a.nz - 1 ? at(ix, iy, iz + 1) : s0;
        const T xm = ix > 0 ? at(ix - 1, iy, iz) : s0;
        const T xp = ix < a.nx - 1 ? at(ix + 1, iy, iz) : s0;
        const T ym = iy > 0 ? at(ix, iy - 1, iz) : s0;
        const T yp = iy < a.ny - 1 ? at(ix, iy + 1, iz) : s0;
        __builtin_amdgcn_s_setprio(0);
        write_node(a, ix, iy, iz, s0, grad1(xm, s0, xp, ix, a.nx, a.cx), grad1(ym, s0, yp, iy, a.ny, a.cy),
                   grad1(zm, s0, zp, iz, a.nz, a.cz));
        zm = s0;
        s0 = zp;
    }
}

// Plane forms of the node field for the tracer's cell cache: node (ix, iy,
// iz) gets the bilinear form of the z-plane cell whose lower corner it is,
//   A = f00, B = f10 - f00, C = f01 - f00, E = (f11 - f01) - B,
// so that f(tx, ty) = A + B tx + C ty + E tx ty on that plane (the last
// column and row, which start no cell, get A = f and B = C = E = 0).  The
// subtractions are those the tracer would do per cell, so the forms equal
// the ones it forms itself, bit for bit.  One thread per output float4
// (component j = t % 4 of node t / 4), so a wave's stores are one contiguous
// 1 KiB run; the neighbour loads hit L1 / L2.  Algorithmic traffic: 16 B read
// + 64 B written per node.
__device__ __forceinline__ void plane_form(const float4 *__restrict__ f, float4 *__restrict__ out, int nx, int ny,
                                           int64_t t) {
    const int j = (int)(t & 3);
    const int64_t i = t >> 2;
    const int ix = (int)(i % nx);
    const int iy = (int)((i / nx) % ny);
    const float4 a = f[i];
    float4 o = a;
    if (j > 0) {
        o = make_float4(0.f, 0.f, 0.f, 0.f);
        if (ix < nx - 1 && iy < ny - 1) {
            const float4 f10 = f[i + 1], f01 = f[i + nx];
            const float4 b = make_float4(f10.x - a.x, f10.y - a.y, f10.z - a.z, f10.w - a.w);
            if (j == 1) {
                o = b;
            } else if (j == 2) {
                o = make_float4(f01.x - a.x, f01.y - a.y, f01.z - a.z, f01.w - a.w);
            } else {
                const float4 f11 = f[i + nx + 1];
                o = make_float4((f11.x - f01.x) - b.x, (f11.y - f01.y) - b.y, (f11.z - f01.z) - b.z,
                                (f11.w - f01.w) - b.w);
            }
        }
    }
    // streamed to HBM (nontemporal): written once, read by the tracer later
    __builtin_nontemporal_store((f32x4){o.x, o.y, o.z, o.w}, reinterpret_cast<f32x4 *>(out + t));
}

__global__ __launch_bounds__(256) void plane_forms_kernel(const float4 *__restrict__ f, float4 *__restrict__ out,
                                                          int nx, int ny, int64_t n4) {
    // grid-stride: a launch holds fewer than 2^32 work-items
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n4; t += (int64_t)gridDim.x * blockDim.x)
        plane_form(f, out, nx, ny, t);
}

template <typename T>
int launch(const void *field, int64_t sx, int64_t sy, int64_t sz, const tt_grid *g, double alpha, double beta,
           double ne_max, double k0, const double *sumsq, int64_t count, float *out4, hipStream_t st) {
    GradArgs<T> a;
    a.f = static_cast<const T *>(field);
    a.sx = sx;
    a.sy = sy;
    a.sz = sz;
    a.nx = g->nx;
    a.ny = g->ny;
    a.nz = g->nz;
    a.beta = (T)beta;
    a.clipv = (T)(ne_max - alpha);
    a.alpha = alpha;
    a.cx = (T)(-0.5 * g->dz / (2.0 * g->dx));
    a.cy = (T)(-0.5 * g->dz / (2.0 * g->dy));
    a.cz = (T)(-0.5 * g->dz / (2.0 * g->dz));
    a.phase_scale = (float)(k0 * g->dz);
    a.sumsq = sumsq;
    a.count = (double)count;
    a.out = reinterpret_cast<float4 *>(out4);
    // The input's contiguous axis, by its strides: any strides are right on any path.
    const auto mag = [](int64_t v) { return v < 0 ? -v : v; };
    const bool bz = mag(sz) < mag(sy) && mag(sz) < mag(sx), fx = !bz && mag(sx) <= mag(sy);
    const int tx = fx ? 64 : 32, tb = 1024 / tx;
    const int nb = bz ? g->nz : g->ny;
    // The longest runs, up to `longest`, that still give `enough` blocks.
    const auto shape = [&](int bx, int bb, int nbb, int nc, int longest, int enough) {
        const int64_t tiles = tt::ceil_div(g->nx, bx) * tt::ceil_div(nbb, bb);
        a.run = longest;
        while (a.run > 2 && tiles * tt::ceil_div(nc, a.run) < enough) a.run /= 2;
        return dim3((unsigned)tt::ceil_div(g->nx, bx), (unsigned)tt::ceil_div(nbb, bb),
                    (unsigned)tt::ceil_div(nc, a.run));
    };
    // On a few planes along b most of a tile is empty: 1024 x 1024 x 3 fp32 13 us by
    // columns and 45 by tiles (z fastest, x next), x 6 32 and 46, x 8 76 and 47; with
    // x fastest 1024 x 8 x 1024 fp64 46 and 50.  Columns of an input with z fastest
    // and x slowest lie far apart: x 3 41 and 46, x 4 53 and 45 (300 x 300 x 4 8.2 and 10.4).
    if (nb <= (fx ? 8 : bz && mag(sx) > mag(sy) ? 4 : 6)) {
        const dim3 grid = shape(64, 4, g->ny, g->nz, 16, bz ? 1 : 2048);
        hipLaunchKernelGGL(grad_columns_kernel<T>, grid, dim3(256), 0, st, a);
        TT_LAUNCH_CHECK("tt_grad_stencil launch");
        return TT_OK;
    }
    // Runs of 32 planes (64 at 512^3: 544 us); on smaller grids shorter ones, which
    // give more blocks and read their two planes of halo more often: about five
    // blocks a CU, four where lanes run along x, and half of that in fp64.
    const int enough = !fx ? 1280 : sizeof(T) == 4 ? 1024 : 512;
    const dim3 grid = shape(tx, tb, nb, bz ? g->ny : g->nz, 32, enough);
    if (bz)
        hipLaunchKernelGGL((grad_kernel<T, 32, true, false>), grid, dim3(256), 0, st, a);
    else if (fx)
        hipLaunchKernelGGL((grad_kernel<T, 64, false, true>), grid, dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((grad_kernel<T, 32, false, false>), grid, dim3(256), 0, st, a);
    TT_LAUNCH_CHECK("tt_grad_stencil launch");
    return TT_OK;
}

}  // namespace

extern "C" int tt_grad_stencil(const void *field, int32_t dtype, int64_t sx, int64_t sy, int64_t sz,
                               const tt_grid *grid, double alpha, double beta, double ne_max, double k0,
                               const double *sumsq, int64_t count, float *out4, void *stream) {
    TT_REQUIRE(field && grid && out4, "tt_grad_stencil: null pointer");
    TT_REQUIRE(grid->nx >= 2 && grid->ny >= 2 && grid->nz >= 2,
               "tt_grad_stencil: every axis needs >= 2 nodes (np.gradient), got %d x %d x %d", grid->nx,
               grid->ny, grid->nz);
    TT_REQUIRE(grid->nz <= 65535, "tt_grad_stencil: nz > 65535");
    TT_REQUIRE(grid->dx > 0 && grid->dy > 0 && grid->dz > 0, "tt_grad_stencil: spacing must be > 0");
    TT_REQUIRE(!sumsq || count > 0, "tt_grad_stencil: count must be > 0 with sumsq");
    hipStream_t st = tt::as_stream(stream);
    if (dtype == 0) return launch<float>(field, sx, sy, sz, grid, alpha, beta, ne_max, k0, sumsq, count, out4, st);
    if (dtype == 1) return launch<double>(field, sx, sy, sz, grid, alpha, beta, ne_max, k0, sumsq, count, out4, st);
    tt::set_error("tt_grad_stencil: dtype must be 0 (float32) or 1 (float64), got %d", dtype);
    return TT_ERR_ARG;
}

extern "C" int tt_plane_forms(const float *field4, const tt_grid *grid, float *forms, void *stream) {
    TT_REQUIRE(field4 && grid && forms, "tt_plane_forms: null pointer");
    TT_REQUIRE(grid->nx >= 2 && grid->ny >= 2 && grid->nz >= 1, "tt_plane_forms: grid needs >= 2 nodes in x and y");
    TT_REQUIRE(forms != field4, "tt_plane_forms: forms must not alias field4");
    const int64_t n4 = 4 * (int64_t)grid->nx * grid->ny * grid->nz;
    const int64_t blocks = std::min<int64_t>(tt::ceil_div(n4, 256), (int64_t)1 << 22);
    hipLaunchKernelGGL(plane_forms_kernel, dim3((unsigned)blocks), dim3(256), 0,
                       tt::as_stream(stream), reinterpret_cast<const float4 *>(field4),
                       reinterpret_cast<float4 *>(forms), grid->nx, grid->ny, n4);
    TT_LAUNCH_CHECK("tt_plane_forms launch");
    return TT_OK;
}
