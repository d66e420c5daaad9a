// Detectors: the ray-transfer optics and Rays.histogram of
// particle_tracking/ray_transfer_matrix.py (RTM:37-154, 173-191, 208-299).
//
// Each ray's [x, theta, y, phi] goes through the optical train in fp64
// registers (a 4x4 block-diagonal matrix per element is two scalar updates;
// rejected rays become NaN, RTM:77-78), then into one or more histograms.
// Binning follows np.histogram2d exactly: edges e_i = i*step + min with
// step = (max - min)/n (np.linspace), bin = searchsorted(e, v, 'right') - 1,
// v == max counts in the last bin, outside values and NaN are dropped.
// Histograms are stored transposed, H[iy][ix] (RTM:191).
//
// Counts are uint32 atomics (order-independent, bit-reproducible);
// interferogram weights are float32 atomics.  Each workgroup first bins its
// 512 rays into a private LDS copy of the bin window they touch when that
// window is small (rays sorted by entry column land close together on the
// detector), then flushes the non-zero bins; otherwise it adds to global
// memory directly.
#include <algorithm>

#include "launch_shape.h"
#include "tt_internal.h"

#pragma clang fp contract(off)

namespace {

struct DetDev {
    int32_t n_ops, to_mm, mode;
    int32_t again;  // the train and bins are those of the detector before
    tt_optic ops[TT_MAX_OPS];
    int32_t nbx, nby;
    double xmin, xmax, ymin, ymax, xstep, ystep, xinv, yinv;
    double tilt_k;
    uint32_t *counts;
    float *wsum;
};

struct DetArgs {
    DetDev d[TT_MAX_DETECTORS];
    int32_t ndet;
    const double *rf;
    int64_t ld, n;
    const double *phase;
};

// apply the train; returns false when the ray is rejected (or NaN)
__device__ __forceinline__ bool apply_train(const DetDev &d, double &x, double &th, double &y, double &ph) {
    if (d.to_mm) {
        x = x * 1e3;
        y = y * 1e3;
    }
    for (int i = 0; i < d.n_ops; ++i) {
        const tt_optic o = d.ops[i];
        switch (o.op) {
            case TT_OP_DISTANCE:
                x = x + o.a * th;
                y = y + o.a * ph;
                break;
            case TT_OP_LENS:
                th = o.a * x + th;  // a, b: -1 / f (fill_train)
                ph = o.b * y + ph;
                break;
            case TT_OP_APERTURE:
                if (x * x + y * y > o.a * o.a) return false;
                break;
            case TT_OP_STOP:
                if (x * x + y * y < o.a * o.a) return false;
                break;
            case TT_OP_KNIFE: {
                const double v = o.axis == 2 ? y : x;
                if ((o.b > 0 && v > o.a) || (o.b < 0 && v < o.a)) return false;
                break;
            }
            case TT_OP_RECT:
                if (x * x > o.a * o.a && y * y > o.b * o.b) return false;
                break;
            case TT_OP_ANNULUS: {
                const double r2 = x * x + y * y;
                if (r2 > o.a * o.a && r2 < o.b * o.b) return false;
                break;
            }
            default:
                break;
        }
    }
    return !(isnan(x) || isnan(th) || isnan(y) || isnan(ph));
}

// np.histogram(bins=n, range=(lo, hi)) bin of v, or -1 if dropped
__device__ __forceinline__ int bin_of(double v, double lo, double hi, double step, double inv, int n) {
    if (!(v >= lo && v <= hi)) return -1;
    if (v == hi) return n - 1;
    int b = (int)((v - lo) * inv);  // near enough for the edges below to decide
    b = b < 0 ? 0 : (b > n - 1 ? n - 1 : b);
    // correct against the exact np.linspace edges (i*step + lo; last = hi)
    while (b > 0 && v < (double)b * step + lo) --b;
    while (b < n - 1 && v >= ((b + 1 == n) ? hi : (double)(b + 1) * step + lo)) ++b;
    return b;
}

constexpr int kDetBlock = 512;  // a ray a thread
constexpr int kLdsBins = 8192;  // private window: 32 KB of uint32/float

using tt::lds_barrier;

__device__ __forceinline__ int wave_min(int v) {
    for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ int wave_max(int v) {
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    return v;
}

// A ray carried to a detector: where it meets it and its bin there (bx < 0: none)
struct Hit {
    double x;
    int bx, by;
};
__device__ __forceinline__ Hit hit(const DetDev &d, bool live, double x, double th, double y, double ph) {
    Hit h{0.0, -1, -1};
    if (live && apply_train(d, x, th, y, ph)) {
        h.bx = bin_of(x, d.xmin, d.xmax, d.xstep, d.xinv, d.nbx);
        h.by = bin_of(y, d.ymin, d.ymax, d.ystep, d.yinv, d.nby);
    }
    h.x = x;
    if (h.by < 0) h.bx = -1;
    return h;
}
__device__ __forceinline__ float weight(const DetDev &d, double phase, double x) {
    return (float)(1.0 + cos(phase - d.tilt_k * x));
}

// A block takes its rays through each detector in turn: the bin window of its
// hits (wave reductions, then 4 LDS atomics per wave), a private LDS copy of
// that window when it holds at most kLdsBins bins, then the non-zero bins
// flushed with global atomics.  The barriers order LDS only, so the flush of one
// detector overlaps the next.  Detectors of one train and one set of bins follow
// each other (tt_detect) and share positions, bins and window.
// Bound by the latency of that chain, not by the atomics (with them left out it
// takes 2 to 15% less): short chains on many waves.  1e7 sorted rays on three
// detectors of 2048^2 (a shadowgram and an interferogram of the same optics, a
// schlieren image) 590 -> 371 us, 1e5 on 512^2 55 -> 20, 1e6 in launch order 155
// -> 135, as 256 threads of four rays each with the train of every detector and
// fp64 quotients for lenses and bins before; 256 threads of two rays 356, 31 and
// 143.
__global__ __launch_bounds__(kDetBlock) void detect_kernel(DetArgs a) {
    __shared__ uint32_t lds[kLdsBins];
    __shared__ int win[4];  // bx0, bx1, by0, by1 of this block's hits
    const int64_t i = ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * kDetBlock + threadIdx.x;
    const bool live = i < a.n;
    double x0 = 0.0, th0 = 0.0, y0 = 0.0, ph0 = 0.0, phase = 0.0;
    if (live) {
        x0 = a.rf[i];
        th0 = a.rf[a.ld + i];
        y0 = a.rf[2 * a.ld + i];
        ph0 = a.rf[3 * a.ld + i];
        if (a.phase) phase = a.phase[i];
    }
    const auto clear_window = [&] {
        if (threadIdx.x == 0) {
            win[0] = 0x7fffffff;
            win[1] = -1;
            win[2] = 0x7fffffff;
            win[3] = -1;
        }
    };
    clear_window();
    Hit h{0.0, -1, -1};
    int wx0 = 0, wy0 = 0, ww = 0;
    int64_t area = 0;
    for (int k = 0; k < a.ndet; ++k) {
        const DetDev &d = a.d[k];
        lds_barrier();  // win is cleared; the previous detector's LDS flush reads are done
        if (!d.again) {
            h = hit(d, live, x0, th0, y0, ph0);
            const int bx = h.bx, by = h.by;
            const int lx0 = wave_min(bx >= 0 ? bx : 0x7fffffff), lx1 = wave_max(bx);
            const int ly0 = wave_min(bx >= 0 ? by : 0x7fffffff), ly1 = wave_max(bx >= 0 ? by : -1);
            if ((threadIdx.x & 63) == 0 && lx1 >= 0) {
                atomicMin(&win[0], lx0);
                atomicMax(&win[1], lx1);
                atomicMin(&win[2], ly0);
                atomicMax(&win[3], ly1);
            }
            lds_barrier();
            wx0 = win[0];
            wy0 = win[2];
            ww = win[1] - wx0 + 1;
            area = win[1] >= wx0 ? (int64_t)ww * (win[3] - wy0 + 1) : 0;
        }
        const int bx = h.bx, by = h.by;
        float w = 1.0f;
        if (d.mode == 1 && bx >= 0) w = weight(d, phase, h.x);
        if (area > 0 && area <= kLdsBins) {
            for (int j = threadIdx.x; j < area; j += kDetBlock) lds[j] = 0u;
            lds_barrier();
            if (bx >= 0) {
                const int q = (by - wy0) * ww + (bx - wx0);
                if (d.mode == 1)
                    atomicAdd(reinterpret_cast<float *>(&lds[q]), w);
                else
                    atomicAdd(&lds[q], 1u);
            }
            lds_barrier();
            for (int j = threadIdx.x; j < area; j += kDetBlock) {
                const uint32_t v = lds[j];
                if (v == 0u) continue;
                const int64_t gi = (int64_t)(wy0 + j / ww) * d.nbx + (wx0 + j % ww);
                if (d.mode == 1)
                    atomicAdd(&d.wsum[gi], __uint_as_float(v));
                else
                    atomicAdd(&d.counts[gi], v);
            }
        } else if (bx >= 0) {
            const int64_t gi = (int64_t)by * d.nbx + bx;
            if (d.mode == 1)
                atomicAdd(&d.wsum[gi], w);
            else
                atomicAdd(&d.counts[gi], 1u);
        }
        lds_barrier();  // every thread has read win
        clear_window();
    }
}

__global__ __launch_bounds__(256) void optics_kernel(DetDev d, const double *rin, int64_t ldi, int64_t n,
                                                     double *rout, int64_t ldo) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double x = rin[i], th = rin[ldi + i], y = rin[2 * ldi + i], ph = rin[3 * ldi + i];
    const bool ok = apply_train(d, x, th, y, ph);
    const double nanv = __longlong_as_double(0x7ff8000000000000ll);
    rout[i] = ok ? x : nanv;
    rout[ldo + i] = ok ? th : nanv;
    rout[2 * ldo + i] = ok ? y : nanv;
    rout[3 * ldo + i] = ok ? ph : nanv;
}

// Many rays on few bins: a block keeps the histograms of all detectors in LDS, takes
// rays in strides of the grid and adds each bin to memory once.  In detect_kernel
// every 512 rays add their window's bins; those of rays in launch order are the
// whole detector, and the adds wait for each other at its few addresses.
// 1e7 rays in launch order on one detector of 16^2 150 us (543 by windows; 330 with
// 1024 rays a block there), 128^2 175 (307, 284), three of 64^2 317 (988, 681), of
// 90^2 in two launches 364 (1097, 735), of 128^2 in three 562 (967, 844); sorted 134,
// 172, 273, 327 and 508 (191, 197, 558, 556 and 554 with 1024 rays a block; the last
// 342 by windows).
// From kWholeRays rays a bin on: with fewer a block's own bins outweigh its rays
// (1e6 rays on 64^2 30 us sorted and 34 in launch order, 21 and 49 by windows; on 90^2
// 55 and 57, 21 and 50).  Four blocks a CU as far as LDS lets (two: 10% slower).
constexpr int kWholeBins = 16384;  // of a launch's detectors: 64 KB
constexpr int kWholeRays = 200;
extern __shared__ uint32_t whole[];
__global__ __launch_bounds__(kDetBlock) void detect_whole_kernel(DetArgs a, int bins) {
    for (int j = threadIdx.x; j < bins; j += kDetBlock) whole[j] = 0u;
    lds_barrier();
    for (int64_t i = (int64_t)blockIdx.x * kDetBlock + threadIdx.x; i < a.n; i += (int64_t)gridDim.x * kDetBlock) {
        const double x = a.rf[i], th = a.rf[a.ld + i], y = a.rf[2 * a.ld + i], ph = a.rf[3 * a.ld + i];
        const double phase = a.phase ? a.phase[i] : 0.0;
        Hit h{0.0, -1, -1};
        int first = 0;
        for (int k = 0; k < a.ndet; ++k) {
            const DetDev &d = a.d[k];
            if (!d.again) h = hit(d, true, x, th, y, ph);
            if (h.bx >= 0) {
                const int q = first + h.by * d.nbx + h.bx;
                if (d.mode == 1)
                    atomicAdd(reinterpret_cast<float *>(&whole[q]), weight(d, phase, h.x));
                else
                    atomicAdd(&whole[q], 1u);
            }
            first += d.nbx * d.nby;
        }
    }
    lds_barrier();
    int first = 0;
    for (int k = 0; k < a.ndet; ++k) {
        const DetDev &d = a.d[k];
        const int n = d.nbx * d.nby;
        for (int j = threadIdx.x; j < n; j += kDetBlock) {
            const uint32_t v = whole[first + j];
            if (v == 0u) continue;
            if (d.mode == 1)
                atomicAdd(&d.wsum[j], __uint_as_float(v));
            else
                atomicAdd(&d.counts[j], v);
        }
        first += n;
    }
}

int fill_train(const tt_train *t, DetDev &d) {
    TT_REQUIRE(t, "null optical train");
    TT_REQUIRE(t->n_ops >= 0 && t->n_ops <= TT_MAX_OPS, "optical train has %d ops (max %d)", t->n_ops, TT_MAX_OPS);
    d.n_ops = t->n_ops;
    d.to_mm = t->to_mm;
    for (int i = 0; i < t->n_ops; ++i) {
        const tt_optic &o = t->ops[i];
        TT_REQUIRE(o.op >= TT_OP_DISTANCE && o.op <= TT_OP_ANNULUS, "optical op %d: unknown code %d", i, o.op);
        if (o.op == TT_OP_LENS) TT_REQUIRE(o.a != 0 && o.b != 0, "optical op %d: lens focal length 0", i);
        if (o.op == TT_OP_KNIFE) {
            TT_REQUIRE(o.axis == 0 || o.axis == 2, "optical op %d: knife edge axis must be 0 (x) or 2 (y)", i);
            TT_REQUIRE(o.b != 0, "optical op %d: knife edge direction must be <0 or >0", i);
        }
        d.ops[i] = o;
        if (o.op == TT_OP_LENS) {
            d.ops[i].a = -1.0 / o.a;
            d.ops[i].b = -1.0 / o.b;
        }
    }
    return TT_OK;
}

}  // namespace

extern "C" int tt_optics_apply(const tt_train *train, const double *r_in, int64_t ld_in, int64_t n, double *r_out,
                               int64_t ld_out, void *stream) {
    DetDev d{};
    int rc = fill_train(train, d);
    if (rc) return rc;
    TT_REQUIRE(n >= 0 && ld_in >= n && ld_out >= n, "tt_optics_apply: bad sizes");
    if (n == 0) return TT_OK;
    TT_REQUIRE(r_in && r_out, "tt_optics_apply: null pointer");
    hipLaunchKernelGGL(optics_kernel, dim3((unsigned)tt::ceil_div(n, 256)), dim3(256), 0, tt::as_stream(stream), d,
                       r_in, ld_in, n, r_out, ld_out);
    TT_LAUNCH_CHECK("tt_optics_apply launch");
    return TT_OK;
}

extern "C" int tt_detect(const tt_detector *dets, int32_t ndet, const double *rf, int64_t ld, const double *phase,
                         int64_t n, void *stream) {
    TT_REQUIRE(dets && ndet >= 1 && ndet <= TT_MAX_DETECTORS, "tt_detect: need 1..%d detectors", TT_MAX_DETECTORS);
    TT_REQUIRE(n >= 0 && ld >= n, "tt_detect: bad sizes");
    if (n == 0) return TT_OK;
    TT_REQUIRE(rf, "tt_detect: null rays");
    DetArgs a{};
    for (int k = 0; k < ndet; ++k) {
        const tt_detector &s = dets[k];
        DetDev &d = a.d[k];
        int rc = fill_train(&s.train, d);
        if (rc) return rc;
        const tt_hist &h = s.hist;
        TT_REQUIRE(h.nbx >= 1 && h.nby >= 1, "tt_detect: detector %d has no bins", k);
        TT_REQUIRE(h.xmax > h.xmin && h.ymax > h.ymin, "tt_detect: detector %d has an empty range", k);
        TT_REQUIRE(s.mode == 0 || s.mode == 1, "tt_detect: detector %d mode must be 0 or 1", k);
        TT_REQUIRE(s.mode == 0 ? s.counts != nullptr : s.wsum != nullptr, "tt_detect: detector %d output is null", k);
        TT_REQUIRE(s.mode == 0 || phase, "tt_detect: interferogram needs the phase");
        d.mode = s.mode;
        d.nbx = h.nbx;
        d.nby = h.nby;
        d.xmin = h.xmin;
        d.xmax = h.xmax;
        d.ymin = h.ymin;
        d.ymax = h.ymax;
        d.xstep = (h.xmax - h.xmin) / h.nbx;
        d.ystep = (h.ymax - h.ymin) / h.nby;
        d.xinv = 1.0 / d.xstep;
        d.yinv = 1.0 / d.ystep;
        d.tilt_k = s.tilt_k;
        d.counts = s.counts;
        d.wsum = s.wsum;
    }
    // detectors of one train and one set of bins follow each other: their rays
    // are carried to the detector and binned once (a shadowgram and the
    // interferogram of the same optics)
    const auto same = [](const DetDev &p, const DetDev &q) {
        if (p.n_ops != q.n_ops || p.to_mm != q.to_mm || p.nbx != q.nbx || p.nby != q.nby || p.xmin != q.xmin ||
            p.xmax != q.xmax || p.ymin != q.ymin || p.ymax != q.ymax)
            return false;
        for (int i = 0; i < p.n_ops; ++i)
            if (p.ops[i].op != q.ops[i].op || p.ops[i].axis != q.ops[i].axis || p.ops[i].a != q.ops[i].a ||
                p.ops[i].b != q.ops[i].b)
                return false;
        return true;
    };
    for (int k = 1; k < ndet; ++k)
        for (int j = k - 1; j >= 0; --j)
            if (same(a.d[j], a.d[k])) {
                std::rotate(a.d + j + 1, a.d + k, a.d + k + 1);
                a.d[j + 1].again = 1;
                break;
            }
    a.ndet = ndet;
    a.rf = rf;
    a.ld = ld;
    a.n = n;
    a.phase = phase;
    // groups of detectors that detect_whole_kernel takes at once, if it takes them all
    int group[TT_MAX_DETECTORS], count[TT_MAX_DETECTORS], groups = 0;
    for (int k = 0; k < ndet && groups >= 0; ++k) {
        const int64_t bins = (int64_t)a.d[k].nbx * a.d[k].nby;
        const bool more = groups > 0 && group[groups - 1] + bins <= kWholeBins;
        if (!more) group[groups] = count[groups] = 0, ++groups;
        ++count[groups - 1];
        if (bins > kWholeBins || n < kWholeRays * (group[groups - 1] += (int)bins)) groups = -1;
    }
    if (groups > 0) {
        for (int g = 0, k = 0; g < groups; k += count[g], ++g) {
            DetArgs w = a;
            w.ndet = count[g];
            std::copy(a.d + k, a.d + k + count[g], w.d);
            w.d[0].again = 0;
            // resident at once, each with as many rays as bins to add at least, and with
            // 1024, so that fewer partial sums of weights meet in a bin than by windows
            const int64_t blocks = std::min<int64_t>(256 * std::min(4, kWholeBins * 5 / 2 / group[g]),
                                                     tt::ceil_div(n, (int64_t)std::max(2 * kDetBlock, group[g])));
            hipLaunchKernelGGL(detect_whole_kernel, dim3((unsigned)blocks), dim3(kDetBlock),
                               (size_t)group[g] * sizeof(uint32_t), tt::as_stream(stream), w, group[g]);
            TT_LAUNCH_CHECK("tt_detect launch");
        }
        return TT_OK;
    }
    const tt::Blocks b = tt::spread(tt::ceil_div(n, (int64_t)kDetBlock), kDetBlock);
    hipLaunchKernelGGL(detect_kernel, dim3(b.x, b.y), dim3(kDetBlock), 0, tt::as_stream(stream), a);
    TT_LAUNCH_CHECK("tt_detect launch");
    return TT_OK;
}
