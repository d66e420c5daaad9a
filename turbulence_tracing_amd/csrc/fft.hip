// Gaussian random field by inverse 3-D FFT: the work of gaussian3D_FFT
// (gaussian_fields/turboGen.py:488-538), restructured for the GPU.
//
// The spectrum F(k) = [Wr(c) + Wr(c') + i (Wi(c) - Wi(c'))] sqrt(P(k)) is
// Hermitian (c' is the centred-grid partner of c, the np.flip of TG:525-526
// for odd sizes and the index of -k for any size), so the real output
// ifftn(F).real is produced from the half spectrum kx in [0, nx/2]:
//   pass Z: generate F (noise x sqrt P, zero mode, TG:522-534) for a block of
//           kx columns directly into LDS and inverse-FFT along z;
//   pass Y: inverse-FFT along y;
//   pass X: complete each row by Hermitian symmetry, inverse-FFT along x,
//           keep the real part times 1/(nx ny nz) (numpy's ifftn scale) and
//           reduce the sum of squares for the unit-RMS normalisation.
// Each pass stages a batch of pencils in LDS and runs a Stockham autosort
// FFT (radix 8/4/2/3/5 butterflies, direct DFT passes for other primes)
// with the twiddle table in LDS.  The spectrum F is never written: pass Z
// writes the z-transformed half spectrum.  Traffic per field:
// 8 (Z) + 16 (Y) + 8 + 4 (X) bytes per half-spectrum element.
#include <climits>
#include <cmath>
#include <vector>

#include "launch_shape.h"
#include "tt_internal.h"

namespace {

constexpr int kThreads = 256;
constexpr int kElems = 32;                     // complex values per thread per pass
constexpr int kBatch = kThreads * kElems;      // complex values per block
constexpr int kMaxRad = 24;
constexpr int kMaxBins = 2048;  // power-spectrum bins (two doubles each in LDS)

struct AxisPlan {
    int n, nrad;
    int rad[kMaxRad];
};

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
    return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 mul_i(float2 a) { return make_float2(-a.y, a.x); }  // * (+i)

// inverse-sign (e^{+2 pi i q r / R}) DFT of R points in registers
template <int R>
__device__ __forceinline__ void dft(float2 *v);

template <>
__device__ __forceinline__ void dft<2>(float2 *v) {
    const float2 a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
}

template <>
__device__ __forceinline__ void dft<4>(float2 *v) {
    const float2 s02 = cadd(v[0], v[2]), d02 = csub(v[0], v[2]);
    const float2 s13 = cadd(v[1], v[3]), d13 = mul_i(csub(v[1], v[3]));
    v[0] = cadd(s02, s13);
    v[2] = csub(s02, s13);
    v[1] = cadd(d02, d13);
    v[3] = csub(d02, d13);
}

template <>
__device__ __forceinline__ void dft<8>(float2 *v) {
    // split into even/odd radix-4 DFTs, then combine with e^{+2 pi i q / 8}
    float2 e[4] = {v[0], v[2], v[4], v[6]};
    float2 o[4] = {v[1], v[3], v[5], v[7]};
    dft<4>(e);
    dft<4>(o);
    const float h = 0.70710678118654752f;
    const float2 w1 = cmul(o[1], make_float2(h, h));
    const float2 w2 = mul_i(o[2]);
    const float2 w3 = cmul(o[3], make_float2(-h, h));
    v[0] = cadd(e[0], o[0]);
    v[4] = csub(e[0], o[0]);
    v[1] = cadd(e[1], w1);
    v[5] = csub(e[1], w1);
    v[2] = cadd(e[2], w2);
    v[6] = csub(e[2], w2);
    v[3] = cadd(e[3], w3);
    v[7] = csub(e[3], w3);
}

template <>
__device__ __forceinline__ void dft<3>(float2 *v) {
    const float c = -0.5f, s = 0.86602540378443865f;  // e^{2 pi i / 3}
    const float2 a = v[0], b = v[1], d = v[2];
    const float2 t = cadd(b, d), u = csub(b, d);
    const float2 m = make_float2(a.x + c * t.x, a.y + c * t.y);
    const float2 su = make_float2(-s * u.y, s * u.x);  // i s (b - d)
    v[0] = cadd(a, t);
    v[1] = cadd(m, su);
    v[2] = csub(m, su);
}

// the same with the last output's product rounded before its difference
__device__ __forceinline__ void dft3_pow(float2 *v) {
#pragma clang fp contract(off)
    const float c = -0.5f, s = 0.86602540378443865f;
    const float2 a = v[0], b = v[1], d = v[2];
    const float2 t = cadd(b, d), u = csub(b, d);
    const float2 m = make_float2(fmaf(c, t.x, a.x), fmaf(c, t.y, a.y));
    v[0] = cadd(a, t);
    v[1] = make_float2(fmaf(-s, u.y, m.x), fmaf(s, u.x, m.y));
    v[2] = make_float2(m.x - -s * u.y, m.y - s * u.x);
}

template <>
__device__ __forceinline__ void dft<5>(float2 *v) {
    const float c1 = 0.30901699437494742f, s1 = 0.95105651629515357f;   // 2 pi / 5
    const float c2 = -0.80901699437494742f, s2 = 0.58778525229247313f;  // 4 pi / 5
    const float2 a = v[0];
    const float2 t1 = cadd(v[1], v[4]), u1 = csub(v[1], v[4]);
    const float2 t2 = cadd(v[2], v[3]), u2 = csub(v[2], v[3]);
    const float2 m1 = make_float2(a.x + c1 * t1.x + c2 * t2.x, a.y + c1 * t1.y + c2 * t2.y);
    const float2 m2 = make_float2(a.x + c2 * t1.x + c1 * t2.x, a.y + c2 * t1.y + c1 * t2.y);
    // i (s1 u1 + s2 u2) and i (s2 u1 - s1 u2)
    const float2 n1 = make_float2(-(s1 * u1.y + s2 * u2.y), s1 * u1.x + s2 * u2.x);
    const float2 n2 = make_float2(-(s2 * u1.y - s1 * u2.y), s2 * u1.x - s1 * u2.x);
    v[0] = make_float2(a.x + t1.x + t2.x, a.y + t1.y + t2.y);
    v[1] = cadd(m1, n1);
    v[4] = csub(m1, n1);
    v[2] = cadd(m2, n2);
    v[3] = csub(m2, n2);
}

// One Stockham pass of radix R over B pencils of length n in LDS (pencil p
// at buf + p*stride).  Every thread first computes all of its butterflies
// into registers, then all write: in-place with two barriers.
template <int R>
__device__ __forceinline__ void pass_r_body(float2 *buf, int n, int stride, int B, int Ns, const float2 *tw) {
    constexpr int NB = (kElems + R - 1) / R;
    float2 v[NB][R];
    const int nbf = n / R;
    const int total = B * nbf;
    const int twstep = n / (Ns * R);
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const int g = threadIdx.x + i * kThreads;
        if (g < total) {
            const int p = g / nbf, b = g - p * nbf;
            const int k = b % Ns;
            const float2 *pb = buf + p * stride;
#pragma unroll
            for (int r = 0; r < R; ++r) v[i][r] = pb[b + r * nbf];
            if (k) {
#pragma unroll
                for (int r = 1; r < R; ++r) v[i][r] = cmul(v[i][r], tw[r * k * twstep]);
            }
            dft<R>(v[i]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const int g = threadIdx.x + i * kThreads;
        if (g < total) {
            const int p = g / nbf, b = g - p * nbf;
            const int k = b % Ns;
            float2 *pb = buf + p * stride + (b / Ns) * Ns * R + k;
#pragma unroll
            for (int q = 0; q < R; ++q) pb[q * Ns] = v[i][q];
        }
    }
    __syncthreads();
}

// ---------------------------------------------------------------------
// Fixed lengths (128, 192, 256, 384, 512, 1024: powers of two times at most
// one 3) with every size known at compile time, so the index arithmetic is shifts and masks, and with the first and
// the last Stockham pass in registers: the first pass reads its butterfly
// inputs straight from the pass's loader (global memory or the generator)
// and the last one hands its outputs straight to the storer, so a pencil
// goes through LDS twice fewer than with LDS-to-LDS passes only.  Radices: 8
// while 8 divides what is left, then 4 or 2, then the odd prime.
template <int N, int NS>
constexpr int radix_at() {
    int m = N / NS, e = 0;
    while (m % 2 == 0) {
        m /= 2;
        ++e;
    }
    if (e >= 3) return 8;
    if (e == 2) return 4;
    if (e == 1) return 2;
    for (int p = 3;; p += 2)
        if (m % p == 0) return p;
}

// butterfly beta of B * NB -> (pencil p, index b); PFAST: p varies fastest
// (pencils are columns of a row-major plane), else b (pencils are rows)
template <int B, int NB, bool PFAST>
__device__ __forceinline__ void split_bf(int beta, int &p, int &b) {
    if (PFAST) {
        p = beta % B;
        b = beta / B;
    } else {
        p = beta / NB;
        b = beta % NB;
    }
}

// first pass (Ns = 1): inputs are elements b + NB r of pencil p
template <int N, bool PFAST, class Load>
__device__ __forceinline__ void first_pass(float2 *buf, Load load) {
    constexpr int R = radix_at<N, 1>(), NB = N / R, B = kBatch / N, TOT = B * NB;
    constexpr int PER = (TOT + kThreads - 1) / kThreads;
    float2 v[PER][R];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int beta = threadIdx.x + i * kThreads;
        if (TOT % kThreads == 0 || beta < TOT) {
            int p, b;
            split_bf<B, NB, PFAST>(beta, p, b);
#pragma unroll
            for (int r = 0; r < R; ++r) v[i][r] = load(p, b + NB * r);
            dft<R>(v[i]);
        }
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int beta = threadIdx.x + i * kThreads;
        if (TOT % kThreads == 0 || beta < TOT) {
            int p, b;
            split_bf<B, NB, PFAST>(beta, p, b);
#pragma unroll
            for (int q = 0; q < R; ++q) buf[p * (N + 1) + R * b + q] = v[i][q];
        }
    }
    __syncthreads();
}

// last pass (Ns = N / R): outputs are elements b + NS q of pencil p
template <int N, int NS, bool PFAST, bool POW, class Store>
__device__ __forceinline__ void last_pass(const float2 *buf, const float2 *tw, Store store) {
    constexpr int R = N / NS, B = kBatch / N, TOT = B * NS;
    constexpr int PER = (TOT + kThreads - 1) / kThreads;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int beta = threadIdx.x + i * kThreads;
        if (TOT % kThreads == 0 || beta < TOT) {
            int p, b;
            split_bf<B, NS, PFAST>(beta, p, b);
            float2 v[R];
#pragma unroll
            for (int r = 0; r < R; ++r) v[r] = buf[p * (N + 1) + b + NS * r];
            if (b) {
#pragma unroll
                for (int r = 1; r < R; ++r) v[r] = cmul(v[r], tw[r * b]);
            }
            if constexpr (POW && R == 3)
                dft3_pow(v);
            else
                dft<R>(v);
#pragma unroll
            for (int q = 0; q < R; ++q) {
                if constexpr (POW)
                    store(i * R + q, v[q]);
                else
                    store(p, b + NS * q, v[q]);
            }
        }
    }
}

template <int N, int NS, bool PFAST, bool POW, class Store>
__device__ __forceinline__ void rest_passes(float2 *buf, const float2 *tw, Store store) {
    constexpr int R = radix_at<N, NS>();
    if constexpr (NS * R == N) {
        last_pass<N, NS, PFAST, POW>(buf, tw, store);
    } else {
        pass_r_body<R>(buf, N, N + 1, kBatch / N, NS, tw);
        rest_passes<N, NS * R, PFAST, POW>(buf, tw, store);
    }
}

// outputs a thread has in the last pass, at most
template <int N, int NS = 1>
constexpr int outputs_of() {
    constexpr int R = radix_at<N, NS>();
    if constexpr (NS * R == N)
        return (kBatch / N * NS + kThreads - 1) / kThreads * R;
    else
        return outputs_of<N, NS * R>();
}
// f(i, p, j) over them, i as the last pass numbers them
template <int N, bool PFAST, int NS = 1, class F>
__device__ __forceinline__ void each_output(F f) {
    constexpr int R = radix_at<N, NS>();
    if constexpr (NS * R == N) {
        constexpr int B = kBatch / N, TOT = B * NS, PER = (TOT + kThreads - 1) / kThreads;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int beta = threadIdx.x + i * kThreads;
            if (TOT % kThreads == 0 || beta < TOT) {
                int p, b;
                split_bf<B, NS, PFAST>(beta, p, b);
#pragma unroll
                for (int q = 0; q < R; ++q) f(i * R + q, p, b + NS * q);
            }
        }
    } else {
        each_output<N, PFAST, NS * R>(f);
    }
}

// the whole transform of the block's B pencils: load(p, j) -> store(p, j, v), or
// (POW) store(i, v) for the thread's i-th output, each_output's numbers
template <int N, bool PFAST, bool POW = false, class Load, class Store>
__device__ __forceinline__ void fft_pow2(float2 *buf, const float2 *tw, Load load, Store store) {
    first_pass<N, PFAST>(buf, load);
    rest_passes<N, radix_at<N, 1>(), PFAST, POW>(buf, tw, store);
}

enum { kGenNative = 0, kGenNoise = 1, kPassY = 2, kPassX = 3, kFwdX = 4, kPowZ = 5 };

struct PassArgs {
    AxisPlan ap;
    const float2 *tw;  // twiddles of this axis, e^{+2 pi i m / n}
    int nx, ny, nz, nxh;
    int lb;        // any length: log2 of the pencils per block
    float2 *spec;  // [nz][ny][nxh]
    // native spectrum
    double aniso, kmin, kmax;
    float half_beta, sqrt_amp;
    uint32_t key0, key1;
    // caller noise
    const float *wr, *wi, *sp;
    // output
    float *out;
    float scale;
    double *sumsq;
    // power spectrum (kFwdX input, kPowZ binning)
    const float *in;
    int mode, nbins;
    double fz_step, fy_step, fx_step;  // 1 / (n dx) per axis (spectrum_3D_scalar frequencies)
    double bin_w, inv_bin_w;           // bin width in |k| (spectrum_3D_scalar)
    double pscale;                     // factor on |F|^2 (compute3Dspectrum: 1 / nt^2, else 1)
    double *hsum, *hcnt;
};

// (j + n/2) mod n and (2 (n/2) - c) mod n for j, c in [0, n): one conditional
// subtraction each instead of an integer division
__device__ __forceinline__ int centred(int j, int n) {
    const int v = j + n / 2;
    return v >= n ? v - n : v;
}
__device__ __forceinline__ int partner(int c, int n) {
    const int v = 2 * (n / 2) - c;
    return v >= n ? v - n : v;
}

// np.fft.fftfreq(n)[j] = j_signed * (1.0 / n)
__device__ __forceinline__ double fftfreq(int j, int n) {
    const int js = (j <= (n - 1) / 2) ? j : j - n;
    return (double)js * (1.0 / (double)n);
}

__device__ __forceinline__ float2 philox_pair(int64_t lin, uint32_t k0, uint32_t k1) {
    const tt::u32x4 r =
        tt::philox4x32_10(tt::u32x4{(uint32_t)lin, (uint32_t)((uint64_t)lin >> 32), tt::kStreamField, 0u}, k0, k1);
    const float u1 = tt::u01f(r.x), u2 = tt::u01f(r.y);
    // Box-Muller on the hardware log2, sqrt and sin / cos (v_sin / v_cos take
    // revolutions, so sin(2 pi u2) is v_sin(u2)); u1, u2 lie in (0, 1) and are
    // never denormal.  Within ~1e-6 of the correctly rounded forms, which cost
    // 15% of the field's time
    const float rad = __builtin_amdgcn_sqrtf(-2.0f * 0.69314718055994531f * __builtin_amdgcn_logf(u1));
    return make_float2(rad * __builtin_amdgcn_cosf(u2), rad * __builtin_amdgcn_sinf(u2));
}

#pragma clang fp contract(off)
__device__ float sqrt_psd_native(const PassArgs &a, int jx, int jy, int jz) {
    const double fx = fftfreq(jx, a.nx), fy = fftfreq(jy, a.ny), fz = fftfreq(jz, a.nz) / a.aniso;
    const double Ka = sqrt((fx * fx + fy * fy) + fz * fz);
    if (!(Ka >= a.kmin && Ka <= a.kmax && Ka > 0.0)) return 0.0f;
    return a.sqrt_amp * __builtin_amdgcn_exp2f(a.half_beta * __builtin_amdgcn_logf((float)Ka));  // Ka^(beta/2)
}
#pragma clang fp contract(on)

template <int MODE>
__device__ __forceinline__ float2 gen(const PassArgs &a, int jx, int jy, int jz) {
    if ((jx | jy | jz) == 0) return make_float2(0.f, 0.f);  // TG:534
    const int cx = centred(jx, a.nx), cy = centred(jy, a.ny), cz = centred(jz, a.nz);
    const int px = partner(cx, a.nx), py = partner(cy, a.ny), pz = partner(cz, a.nz);
    const int64_t lc = ((int64_t)cx * a.ny + cy) * a.nz + cz;
    const int64_t lp = ((int64_t)px * a.ny + py) * a.nz + pz;
    float2 wc, wp;
    float s;
    if (MODE == kGenNative) {
        s = sqrt_psd_native(a, jx, jy, jz);
        if (s == 0.0f) return make_float2(0.f, 0.f);
        wc = philox_pair(lc, a.key0, a.key1);
        wp = philox_pair(lp, a.key0, a.key1);
    } else {
        s = a.sp[lc];
        wc = make_float2(a.wr[lc], a.wi[lc]);
        wp = make_float2(a.wr[lp], a.wi[lp]);
    }
    return make_float2((wc.x + wp.x) * s, (wc.y - wp.y) * s);
}

// ---------------------------------------------------------------------
// Power spectrum of a real field (the estimators of
// gaussian_fields/calculate_spectrum_3d.py:3-59 and cmpspec.py:147-194).
// The passes above run with the inverse sign; for a real field that gives
// conj(fftn(f)), whose |.|^2 is fftn's.  The field is read as rows along x'
// (the reference's last axis, contiguous in C order), so x' / y' / z' are
// the reference's axes 2 / 1 / 0.  Each stored half-spectrum element also
// stands for its mirror (-k), which has the same power, unless kx' is 0 or
// nx'/2.
// Mode 0 (spectrum_3D_scalar): K = sqrt((k0^2 + k1^2) + k2^2) with k_i the
//   fftfreq(M_i, dx) value of axis i; bin b holds bin_w (b) <= K <
//   bin_w (b + 1), the reference's comparisons, for b <= nbins - 2.
// Mode 1 (compute3Dspectrum): shell round(sqrt(v0^2 + v1^2 + v2^2)) of the
//   reference's loop values v_i in range(-M_i // 2, M_i // 2 - 1), so one
//   index per axis, (M_i - 2) // 2, is never visited; power scaled by
//   1 / nt^2 (rh = fftn(r) / nt).
__device__ __forceinline__ int signed_of(int j, int n) { return (j <= (n - 1) / 2) ? j : j - n; }
// the reference loop value of array index j, or INT_MIN when not visited
__device__ __forceinline__ int loop_value(int j, int n) {
    const int hi = n / 2 - 2;
    if (j == (n - 2) / 2) return INT_MIN;
    return j <= hi ? j : j - n;
}

// The bins an element's power goes to: w0 times to b0 and, where its mirror's
// bin is another one, once to b1 (-1: none).
struct Bins {
    int b0, b1;
    uint32_t w0;
};
#pragma clang fp contract(off)
__device__ __forceinline__ Bins bins_of(const PassArgs &a, int jx, int jy, int jz) {
    const bool self_conj = jx == 0 || (a.nx % 2 == 0 && jx == a.nx / 2);
    if (a.mode == 0) {
        const double f0 = (double)signed_of(jz, a.nz) * a.fz_step;
        const double f1 = (double)signed_of(jy, a.ny) * a.fy_step;
        const double f2 = (double)signed_of(jx, a.nx) * a.fx_step;
        const double K = sqrt((f0 * f0 + f1 * f1) + f2 * f2);
        int b = (int)(K * a.inv_bin_w);  // at most one off: corrected by the comparisons
        if (K < (double)b * a.bin_w) --b;
        else if (K >= (double)(b + 1) * a.bin_w) ++b;
        return Bins{b <= a.nbins - 2 ? b : -1, -1, self_conj ? 1u : 2u};
    }
    const auto shell = [&](int ix, int iy, int iz) {
        const int v0 = loop_value(iz, a.nz), v1 = loop_value(iy, a.ny), v2 = loop_value(ix, a.nx);
        if (v0 == INT_MIN || v1 == INT_MIN || v2 == INT_MIN) return -1;
        // round(sqrt(s2)) is the integer b with b (b - 1) < s2 <= b (b + 1)
        const int s2 = v0 * v0 + v1 * v1 + v2 * v2;
        int b = (int)(__builtin_amdgcn_sqrtf((float)s2) + 0.5f);
        if (s2 > b * (b + 1)) ++b;
        if (b > 0 && s2 <= b * (b - 1)) --b;
        return b < a.nbins ? b : -1;
    };
    const int b0 = shell(jx, jy, jz);
    if (self_conj) return Bins{b0, -1, 1u};
    const int b1 = shell(jx ? a.nx - jx : 0, jy ? a.ny - jy : 0, jz ? a.nz - jz : 0);
    return b0 == b1 ? Bins{b0, -1, 2u} : Bins{b0, b1, 1u};
}
#pragma clang fp contract(on)

// A block's histogram.  Lanes next to each other hold neighbouring kx, whose
// power goes to a few bins, and LDS adds to one address wait for each other: so
// lanes spread their adds over up to 16 copies (lane mod copies; as many as the
// FFT's buffer, free by then, has room for), which are summed per tile into the
// block's own.  A block takes several tiles and adds its histogram to the result
// once: those adds go to the same few addresses from every block.  Counts are
// integers in LDS.  Bound by the adds and the bins' arithmetic: pass Z and the two
// before it took 169 us (mode 0) and 188 (mode 1) at 256^3 with adds straight to
// the block's own bins, a tile a block, and a double quotient, root and integer
// remainders an element; 134 and 140 now, 512^3 983 and 1214 -> 888 and 910.
// 512 blocks: two a CU, which is what the tile loop's registers let run (1024:
// 142 and 148; a tile a block 144 and 151).  Two waves a SIMD are asked for: 384
// points, whose 33 outputs a thread take the most registers, would run one (384^3
// 666 and 730 us, with the powers in scratch; 540 and 564 with neither).
constexpr int kPowBlocks = 512;
extern __shared__ __attribute__((aligned(16))) float2 smem[];
struct Histogram {
    // places in LDS, in eight and in four bytes (kept as numbers: through
    // pointers held here the adds become flat ones): the block's sums and
    // counts, the copies' (`stride` apart)
    int hs, hc, cs, cc;
    int nbins, copies, stride;
    double scale;
    static __device__ __forceinline__ double &f64(int at) { return reinterpret_cast<double *>(smem)[at]; }
    static __device__ __forceinline__ uint32_t &u32(int at) { return reinterpret_cast<uint32_t *>(smem)[at]; }
    // own: where the block's histogram begins; spare, bytes: room for copies
    __device__ Histogram(const PassArgs &a, int own, int spare, int bytes)
        : hs(own), hc(2 * (own + a.nbins)), nbins(a.nbins), copies(16), stride(a.nbins | 1), scale(a.pscale) {
        while (copies > 1 && copies * stride * 12 > bytes) copies /= 2;
        cs = copies > 1 ? spare : hs;
        cc = copies > 1 ? 2 * (spare + copies * stride) : hc;
    }
    __device__ void clear_own(int threads) const {
        for (int j = threadIdx.x; j < nbins; j += threads) {
            f64(hs + j) = 0.0;
            u32(hc + j) = 0u;
        }
    }
    __device__ void clear_copies(int threads) const {
        if (copies > 1)
            for (int j = threadIdx.x; j < copies * stride; j += threads) {
                f64(cs + j) = 0.0;
                u32(cc + j) = 0u;
            }
    }
    // power: |F|^2
    __device__ __forceinline__ void add(const Bins &b, float power) const {
        const double p = (double)power * scale;
        const int at = (int)(threadIdx.x & (copies - 1)) * stride;
        if (b.b0 >= 0) {
            atomicAdd(&f64(cs + at + b.b0), b.w0 == 2 ? p + p : p);
            atomicAdd(&u32(cc + at + b.b0), b.w0);
        }
        if (b.b1 >= 0) {
            atomicAdd(&f64(cs + at + b.b1), p);
            atomicAdd(&u32(cc + at + b.b1), 1u);
        }
    }
    __device__ void sum_copies(int threads) const {
        if (copies > 1)
            for (int j = threadIdx.x; j < nbins; j += threads) {
                double t = 0.0;
                uint32_t c = 0;
                for (int k = 0; k < copies; ++k) {
                    t += f64(cs + k * stride + j);
                    c += u32(cc + k * stride + j);
                }
                f64(hs + j) += t;
                u32(hc + j) += c;
            }
    }
    __device__ void flush(const PassArgs &a, int threads) const {
        for (int j = threadIdx.x; j < nbins; j += threads)
            if (const uint32_t c = u32(hc + j)) {
                atomicAdd(&a.hsum[j], f64(hs + j));
                atomicAdd(&a.hcnt[j], (double)c);
            }
    }
};

// add the block's sum of v to *out
template <int THREADS>
__device__ __forceinline__ void block_sum(double v, double *out) {
    __shared__ double red[THREADS / 64];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < THREADS / 64; ++w) t += red[w];
        atomicAdd(out, t);
    }
}

// The fixed lengths: NF points a pencil, kBatch / NF pencils a block.
template <int MODE, int NF>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(MODE == kPowZ ? 2 : 1))) void fft_pass_kernel(PassArgs a) {
    constexpr int BF = kBatch / NF;
    float2 *buf = smem;
    float2 *tw = smem + BF * (NF + 1);
    for (int j = threadIdx.x; j < NF; j += kThreads) tw[j] = a.tw[j];
    if constexpr (MODE == kPowZ) {
        // columns are numbered through the whole spectrum (column q begins at
        // element q of the first plane): only the last tile is ragged
        const int64_t plane = (int64_t)a.nxh * a.ny;
        // The powers of a tile's elements go back to LDS (half of the FFT's
        // buffer, the histogram's copies in the rest): taken from registers, the
        // bins of all of a thread's elements are formed at once in 270 of them.
        float *pw = reinterpret_cast<float *>(buf);
        constexpr int kPw = BF * NF;
        const Histogram H(a, BF * (NF + 1) + NF, kPw / 2, BF * (NF + 1) * 8 - kPw * 4);
        H.clear_own(kThreads);
        for (int64_t first = (int64_t)blockIdx.x * BF; first < plane; first += (int64_t)gridDim.x * BF) {
            float power[outputs_of<NF>()];
            fft_pow2<NF, true, true>(
                buf, tw,
                [&](int p, int j) { return first + p < plane ? a.spec[j * plane + first + p] : make_float2(0.f, 0.f); },
                [&](int i, float2 v) { power[i] = fmaf(v.x, v.x, v.y * v.y); });
            __syncthreads();
            each_output<NF, true>([&](int i, int p, int j) { pw[j * BF + p] = power[i]; });
            H.clear_copies(kThreads);
            __syncthreads();
#pragma unroll 1
            for (int e = threadIdx.x; e < kPw; e += kThreads) {
                const int j = e / BF;
                const uint32_t q = (uint32_t)first + (e - j * BF), ky = q / (uint32_t)a.nxh;
                if (q < (uint32_t)plane) H.add(bins_of(a, (int)(q - ky * a.nxh), (int)ky, j), pw[e]);
            }
            __syncthreads();
            H.sum_copies(kThreads);
            __syncthreads();
        }
        H.flush(a, kThreads);
    } else if constexpr (MODE == kFwdX) {
        const int64_t rows = (int64_t)a.ny * a.nz, r0 = (int64_t)blockIdx.x * BF;
        fft_pow2<NF, false>(
            buf, tw,
            [&](int p, int k) { return make_float2(r0 + p < rows ? a.in[(r0 + p) * NF + k] : 0.f, 0.f); },
            [&](int p, int k, float2 v) {
                if (r0 + p < rows && k < a.nxh) a.spec[(r0 + p) * a.nxh + k] = v;
            });
    } else if constexpr (MODE == kPassX) {
        const int64_t rows = (int64_t)a.ny * a.nz, r0 = (int64_t)blockIdx.x * BF;
        double ss = 0.0;
        fft_pow2<NF, false>(
            buf, tw,
            [&](int p, int k) {
                if (r0 + p >= rows) return make_float2(0.f, 0.f);
                const float2 *srow = a.spec + (r0 + p) * a.nxh;
                if (k < a.nxh) return srow[k];
                const float2 c = srow[NF - k];
                return make_float2(c.x, -c.y);
            },
            [&](int p, int k, float2 v) {
                if (r0 + p >= rows) return;
                const float o = v.x * a.scale;
                a.out[(r0 + p) * NF + k] = o;
                ss += (double)o * (double)o;
            });
        if (a.sumsq) block_sum<kThreads>(ss, a.sumsq);
    } else {  // kGenNative, kGenNoise (pencils along z) and kPassY (along y)
        const int kx0 = blockIdx.x * BF, fixed = blockIdx.y;
        fft_pow2<NF, true>(
            buf, tw,
            [&](int p, int j) {
                const int kx = kx0 + p;
                if (kx >= a.nxh) return make_float2(0.f, 0.f);
                if constexpr (MODE == kPassY)
                    return a.spec[((int64_t)fixed * a.ny + j) * a.nxh + kx];
                else
                    return gen<MODE>(a, kx, fixed, j);
            },
            [&](int p, int j, float2 v) {
                const int kx = kx0 + p;
                if (kx >= a.nxh) return;
                const int64_t idx = (MODE == kPassY) ? ((int64_t)fixed * a.ny + j) * a.nxh + kx
                                                     : ((int64_t)j * a.ny + fixed) * a.nxh + kx;
                a.spec[idx] = v;
            });
    }
}

// ---------------------------------------------------------------------
// Any other length.  A block takes PB pencils (a power of two, 16 up to 309
// points, more of short ones) in LDS as [element][pencil], two copies of them, and each Stockham
// pass goes from one to the other: one barrier a pass, and any number of
// butterflies a thread.  Lanes run over pencils first, so neighbouring lanes
// share a butterfly: its twiddles are LDS broadcasts, and the columns of passes
// Y and Z are read and written 128 bytes at a time.  Pencils are numbered
// through the whole spectrum (not per plane), so only the last block is ragged.
// The pencil index is XORed with the element's low bits but the last, so that
// reading along a pencil (pass X loads and stores rows) meets different banks
// too and two neighbouring pencils stay one aligned 16-byte read.
// Quotients of small integers are taken in fp32 (exact below 2^21).
//
// A prime factor R > 5 is a DFT of R points by definition.  A thread computes
// kQ consecutive outputs of kP pencils: a term's inputs are read once for kQ
// outputs and its factors e^{2 pi i q r / R} (from the twiddle table, at q r mod
// R) once for kP pencils, so (with kQ = 4) 8 complex products go with 5 LDS
// reads.  The terms are added in order of r: the same bits as one output per
// thread with two reads a term, as which it was bound by LDS (201^3 = 3 x 67:
// 1610 us, here 289; 257^3 5700, here 1730); now it is bound by the products'
// issue.  (With the inputs folded by the symmetry of the factors, on
// v_mfma_f32_16x16x4_f32, they took 162 and 492 us, but sums in that order move
// the field's rounding: its sum of squares by more than 1e-9.)  Lengths without
// such a factor gain from the rest: 300^3 620 -> 317 us, 64^3 85 -> 17 us.
// 512 threads a block: with 256, 300^3 took 457 us.  Six waves a SIMD: left to
// itself the compiler takes more registers and 201^3 took 350.
constexpr int kAnyThreads = 512;
__device__ __forceinline__ int fdiv(int v, float inv) { return (int)(((float)v + 0.5f) * inv); }
__device__ __forceinline__ int at(int j, int p, int lb) { return (j << lb) + (p ^ (j & (((1 << lb) - 1) & ~1))); }

template <int R>
__device__ __forceinline__ void any_pass(const float2 *in, float2 *out, int n, int lb, int Ns, const float2 *tw) {
    const int nbf = n / R, twstep = nbf / Ns;
    const float iNs = 1.0f / (float)Ns;
    const int p = threadIdx.x & ((1 << lb) - 1);
    for (int b = threadIdx.x >> lb; b < nbf; b += kAnyThreads >> lb) {
        const int hi = fdiv(b, iNs), k = b - hi * Ns;
        float2 v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = in[at(b + r * nbf, p, lb)];
        if (k) {
#pragma unroll
            for (int r = 1; r < R; ++r) v[r] = cmul(v[r], tw[r * k * twstep]);
        }
        dft<R>(v);
        const int o = hi * Ns * R + k;
#pragma unroll
        for (int q = 0; q < R; ++q) out[at(o + q * Ns, p, lb)] = v[q];
    }
}

constexpr int kP = 2;

template <int kQ>
__device__ __forceinline__ void any_pass_prime(const float2 *in, float2 *out, int n, int lb, int Ns, int R,
                                               const float2 *tw) {
    const int nbf = n / R, twstep = nbf / Ns, lg = lb > 1 ? lb - 1 : 0;  // log2 of the pencil groups
    const int tiles = (R + kQ - 1) / kQ, items = (tiles * nbf) << lg;
    const float inbf = 1.0f / (float)nbf, iNs = 1.0f / (float)Ns;
    // byte offsets: a table entry, a row of pencils
    const uint32_t wrap = (uint32_t)n * 8u, row = (uint32_t)nbf << (lb + 3), swz = lb > 0 ? ((1u << lb) - 2u) * 8u : 0u;
    const char *tw0 = reinterpret_cast<const char *>(tw), *in0 = reinterpret_cast<const char *>(in);
    for (int item = threadIdx.x; item < items; item += kAnyThreads) {
        const int grp = item & ((1 << lg) - 1), bq = item >> lg;
        const int qt = fdiv(bq, inbf), b = bq - qt * nbf;
        const int hi = fdiv(b, iNs), k = b - hi * Ns;
        const int p0 = grp * kP;
        float2 acc[kQ][kP];
        uint32_t w[kQ], dw[kQ];  // of entry (q r mod R) nbf, and its step
#pragma unroll
        for (int j = 0; j < kQ; ++j) {
            const int q = min(kQ * qt + j, R - 1);  // spare outputs repeat the last
            w[j] = 0u;
            dw[j] = (uint32_t)(q * nbf) * 8u;
#pragma unroll
            for (int i = 0; i < kP; ++i) acc[j][i] = make_float2(0.f, 0.f);
        }
        uint32_t e8 = (uint32_t)b * 8u, erow = (uint32_t)b << (lb + 3);  // of element b + r nbf
        for (int r = 0; r < R; ++r, e8 += (uint32_t)nbf * 8u, erow += row) {
            float2 x[kP];  // at()
            const char *px = in0 + erow + (((uint32_t)p0 * 8u) ^ (e8 & swz));
            if (lb > 0) {
                static_assert(__alignof__(smem) % sizeof(float4) == 0, "two pencils are read at once");
                const float4 xx = *reinterpret_cast<const float4 *>(px);
                x[0] = make_float2(xx.x, xx.y);
                x[1] = make_float2(xx.z, xx.w);
            } else {
                x[0] = x[1] = *reinterpret_cast<const float2 *>(px);
            }
            if (k) {
                const float2 t = tw[r * k * twstep];
#pragma unroll
                for (int i = 0; i < kP; ++i)
                    x[i] = make_float2(fmaf(x[i].x, t.x, -(x[i].y * t.y)), fmaf(x[i].y, t.x, x[i].x * t.y));
            }
#pragma unroll
            for (int j = 0; j < kQ; ++j) {
                const float2 c = *reinterpret_cast<const float2 *>(tw0 + w[j]);
#pragma unroll
                for (int i = 0; i < kP; ++i) {
                    // spelled out, so that every build rounds alike
                    acc[j][i].x = __fadd_rn(acc[j][i].x, fmaf(x[i].x, c.x, -(x[i].y * c.y)));
                    acc[j][i].y = __fadd_rn(acc[j][i].y, fmaf(x[i].y, c.x, x[i].x * c.y));
                }
                w[j] += dw[j];
                w[j] = min(w[j], w[j] - wrap);  // mod n: the difference wraps to a large value below n
            }
        }
        const int o = hi * Ns * R + k;
#pragma unroll
        for (int j = 0; j < kQ; ++j)
#pragma unroll
            for (int i = 0; i < kP; ++i)
                if (kQ * qt + j < R && i < (1 << lb)) out[at(o + (kQ * qt + j) * Ns, p0 + i, lb)] = acc[j][i];
    }
}

// The outputs per thread, 2 to 6, for which the block's turns over its items
// times the work of a turn (as measured, about kQ + 1) are least: 257 points
// take 520 items of four outputs, so two turns of 512 threads, but 416 of five.
__device__ __forceinline__ int outputs_per_thread(int R, int nbf, int lb) {
    int best = 4, least = 1 << 30;
    for (int q = 2; q <= 6; ++q) {
        const int items = ((R + q - 1) / q * nbf) << (lb > 1 ? lb - 1 : 0);
        const int cost = (items + kAnyThreads - 1) / kAnyThreads * (q + 1);
        if (cost < least) {
            least = cost;
            best = q;
        }
    }
    return best;
}

template <int MODE>
__global__ __launch_bounds__(kAnyThreads) __attribute__((amdgpu_waves_per_eu(6, 6))) void fft_any_kernel(PassArgs a) {
    const int n = a.ap.n, lb = a.lb, PB = 1 << lb;
    float2 *buf = smem, *alt = smem + n * PB, *tw = alt + n * PB;
    for (int j = threadIdx.x; j < n; j += kAnyThreads) tw[j] = a.tw[j];
    // pencils: columns (elements `step` apart from `base`) or rows
    constexpr bool kRows = MODE == kPassX || MODE == kFwdX;
    // Neighbouring columns share the lines that their elements lie in: blocks of
    // neighbouring columns go to one XCD, whose L2 then holds a line for all of
    // them (a block of 4 moves 32 bytes of each, one of 4096 points 8).  Fields of
    // 256 x 1280 x 256 1417 -> 1001 us, 128 x 2048 x 128 701 -> 525, 128 x 4096 x 128
    // 1840 -> 1347, 320^3 380 -> 343.
    const int64_t block = kRows || gridDim.y > 1 ? (int64_t)blockIdx.y * gridDim.x + blockIdx.x
                                                 : tt::xcd_block((int)blockIdx.x, (int)gridDim.x);
    const int64_t first = block * PB;
    const int64_t plane = (int64_t)a.nxh * a.ny;
    const int p0 = threadIdx.x & (PB - 1), j0 = threadIdx.x >> lb, dj = kAnyThreads >> lb;
    const int64_t count = kRows ? (int64_t)a.ny * a.nz : MODE == kPassY ? (int64_t)a.nxh * a.nz : plane;
    if (first >= count) return;  // a spare block of the last row (tt::spread)
    const float in_ = 1.0f / (float)n;
    int kx = 0, ky = 0;
    int64_t base = 0, step = 0;
    const bool live = first + p0 < count;
    if (!kRows) {
        const uint32_t q = live ? (uint32_t)(first + p0) : 0u;
        const uint32_t row = q / (uint32_t)a.nxh;
        kx = (int)(q - row * (uint32_t)a.nxh);
        ky = (int)row;
        step = MODE == kPassY ? a.nxh : plane;
        base = MODE == kPassY ? (int64_t)row * plane + kx : (int64_t)q;
        for (int j = j0; j < n; j += dj) {
            float2 v = make_float2(0.f, 0.f);
            if (live) {
                if constexpr (MODE == kGenNative || MODE == kGenNoise)
                    v = gen<MODE>(a, kx, ky, j);
                else
                    v = a.spec[base + j * step];
            }
            buf[at(j, p0, lb)] = v;
        }
    } else {
        for (int e = threadIdx.x; e < n * PB; e += kAnyThreads) {
            const int p = fdiv(e, in_), k = e - p * n;
            const int64_t row = first + p;
            float2 v = make_float2(0.f, 0.f);
            if (row < count) {
                if constexpr (MODE == kFwdX) {
                    v.x = a.in[row * n + k];
                } else {  // complete the row by Hermitian symmetry
                    const bool mirror = k >= a.nxh;
                    v = a.spec[row * a.nxh + (mirror ? n - k : k)];
                    if (mirror) v.y = -v.y;
                }
            }
            buf[at(k, p, lb)] = v;
        }
    }
    __syncthreads();
    int Ns = 1;
    for (int s = 0; s < a.ap.nrad; ++s) {
        const int R = a.ap.rad[s];
        switch (R) {
            case 8: any_pass<8>(buf, alt, n, lb, Ns, tw); break;
            case 4: any_pass<4>(buf, alt, n, lb, Ns, tw); break;
            case 2: any_pass<2>(buf, alt, n, lb, Ns, tw); break;
            case 3: any_pass<3>(buf, alt, n, lb, Ns, tw); break;
            case 5: any_pass<5>(buf, alt, n, lb, Ns, tw); break;
            default:
                switch (outputs_per_thread(R, n / R, lb)) {
                    case 2: any_pass_prime<2>(buf, alt, n, lb, Ns, R, tw); break;
                    case 3: any_pass_prime<3>(buf, alt, n, lb, Ns, R, tw); break;
                    case 4: any_pass_prime<4>(buf, alt, n, lb, Ns, R, tw); break;
                    case 5: any_pass_prime<5>(buf, alt, n, lb, Ns, R, tw); break;
                    default: any_pass_prime<6>(buf, alt, n, lb, Ns, R, tw); break;
                }
                break;
        }
        Ns *= R;
        __syncthreads();
        float2 *t = buf;
        buf = alt;
        alt = t;
    }
    if constexpr (kRows) {
        double ss = 0.0;
        const int w = MODE == kFwdX ? a.nxh : n;  // elements kept of a row
        const float iw = 1.0f / (float)w;
        for (int e = threadIdx.x; e < w * PB; e += kAnyThreads) {
            const int p = fdiv(e, iw), k = e - p * w;
            const int64_t row = first + p;
            if (row >= count) continue;
            const float2 v = buf[at(k, p, lb)];
            if constexpr (MODE == kFwdX) {
                a.spec[row * a.nxh + k] = v;
            } else {
                const float o = v.x * a.scale;
                a.out[row * n + k] = o;
                ss += (double)o * (double)o;
            }
        }
        if (MODE == kPassX && a.sumsq) block_sum<kAnyThreads>(ss, a.sumsq);
    } else if constexpr (MODE == kPowZ) {
        const Histogram H(a, (2 * PB + 1) * n, (int)(alt - smem), n * PB * 8);
        H.clear_own(kAnyThreads);
        H.clear_copies(kAnyThreads);
        __syncthreads();
        if (live)
            for (int j = j0; j < n; j += dj) {
                const float2 v = buf[at(j, p0, lb)];
                H.add(bins_of(a, kx, ky, j), fmaf(v.x, v.x, v.y * v.y));
            }
        __syncthreads();
        H.sum_copies(kAnyThreads);
        __syncthreads();
        H.flush(a, kAnyThreads);
    } else if (live) {
        for (int j = j0; j < n; j += dj) a.spec[base + j * step] = buf[at(j, p0, lb)];
    }
}

bool fixed_length(int n) { return n == 128 || n == 192 || n == 256 || n == 384 || n == 512 || n == 1024; }

// the passes of a length: 8, then 4 or 2, then the odd primes from the smallest
void factorize(int n, AxisPlan &ap) {
    ap.n = n;
    ap.nrad = 0;
    int m = n;
    int e2 = 0;
    while (m % 2 == 0) {
        m /= 2;
        ++e2;
    }
    while (e2 >= 3) {
        ap.rad[ap.nrad++] = 8;
        e2 -= 3;
    }
    if (e2 == 2) ap.rad[ap.nrad++] = 4;
    if (e2 == 1) ap.rad[ap.nrad++] = 2;
    for (int p = 3; m > 1; p += 2) {
        while (m % p == 0) {
            ap.rad[ap.nrad++] = p;
            m /= p;
        }
    }
}

// LDS of a block: of a fixed length, kBatch / n pencils (padded rows) and the
// twiddles; of any other, two copies of 2^lb pencils and the twiddles
constexpr size_t kMaxLds = 160 * 1024 - 256;  // of 160 KB, some static
size_t smem_fixed(int n) { return ((size_t)kBatch / n * (n + 1) + n) * sizeof(float2); }
size_t smem_any(int n, int lb) { return (((size_t)2 << lb) + 1) * n * sizeof(float2); }
// log2 of the pencils a block takes: 16 while two blocks fit a CU's LDS (up to
// 309 points), then 8, 4 and 2.  One block of 16 alone on a CU leaves it idle
// between its passes: 640^3 took 8360 us with 8 pencils against 4350 with 4 (256
// threads), 320^3 816 with 16 against 465 with 8.  Where 16 short pencils would
// leave most of the 512 threads without an element, more of them, up to 2048
// elements, as long as that leaves 4 blocks a CU: fields of 2048 x 2048 x 4 684 ->
// 300 us, 512 x 512 x 12 76 -> 55, 512 x 48 x 512 169 -> 153 (up to 1024 elements:
// 300, 58 and 169; 32^3 with a quarter of a block a CU 15 -> 19).  At most 256, so
// that a pencil has two threads.
constexpr int kMostPencils = 8;
static_assert(1 << kMostPencils < kAnyThreads, "threads a pencil");
int pencils_any(int n, int64_t count, size_t extra) {
    int lb = 4;
    while (lb < kMostPencils && (n << (lb + 1)) <= 2048 && (count >> (lb + 1)) >= 1024) ++lb;
    while (lb > 1 && smem_any(n, lb) + extra > kMaxLds / 2) --lb;
    while (lb > 0 && smem_any(n, lb) + extra > kMaxLds) --lb;
    return lb;
}

}  // namespace

struct tt_fft_plan_s {
    int nx, ny, nz, nxh;
    AxisPlan ax[3];
    float2 *tw[3];
    float2 *tw_all;
};

extern "C" int tt_fft_plan_create(int32_t nx, int32_t ny, int32_t nz, tt_fft_plan *plan) {
    TT_REQUIRE(plan, "tt_fft_plan_create: null plan pointer");
    TT_REQUIRE(nx >= 2 && ny >= 2 && nz >= 2 && nx <= 4096 && ny <= 4096 && nz <= 4096,
               "tt_fft_plan_create: sizes must be in [2, 4096], got %d x %d x %d", nx, ny, nz);
    tt_fft_plan_s *p = new tt_fft_plan_s();
    p->nx = nx;
    p->ny = ny;
    p->nz = nz;
    p->nxh = nx / 2 + 1;
    const int ns[3] = {nx, ny, nz};
    std::vector<float2> host;
    size_t off[3];
    for (int a = 0; a < 3; ++a) {
        factorize(ns[a], p->ax[a]);
        if (p->ax[a].nrad > kMaxRad) {
            delete p;
            tt::set_error("tt_fft_plan_create: too many factors");
            return TT_ERR_ARG;
        }
        off[a] = host.size();
        for (int m = 0; m < ns[a]; ++m) {
            const double ang = 2.0 * M_PI * (double)m / (double)ns[a];
            host.push_back(make_float2((float)cos(ang), (float)sin(ang)));
        }
    }
    hipError_t e = hipMalloc(&p->tw_all, host.size() * sizeof(float2));
    if (e != hipSuccess) {
        delete p;
        return tt::hip_check(e, "tt_fft_plan_create: hipMalloc");
    }
    e = hipMemcpy(p->tw_all, host.data(), host.size() * sizeof(float2), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        (void)hipFree(p->tw_all);
        delete p;
        return tt::hip_check(e, "tt_fft_plan_create: hipMemcpy");
    }
    for (int a = 0; a < 3; ++a) p->tw[a] = p->tw_all + off[a];
    *plan = p;
    return TT_OK;
}

extern "C" int tt_fft_plan_destroy(tt_fft_plan plan) {
    if (!plan) return TT_OK;
    hipError_t e = hipFree(plan->tw_all);
    delete plan;
    return tt::hip_check(e, "tt_fft_plan_destroy: hipFree");
}

extern "C" int tt_fft_workspace_bytes(tt_fft_plan plan, size_t *bytes) {
    TT_REQUIRE(plan && bytes, "tt_fft_workspace_bytes: null pointer");
    *bytes = (size_t)plan->nz * plan->ny * plan->nxh * sizeof(float2);
    return TT_OK;
}

namespace {

// dynamic LDS above 64 KB must be enabled per kernel
int enable_lds() {
    static int rc = -1;
    if (rc >= 0) return rc;
    const void *any[] = {(const void *)fft_any_kernel<kGenNative>, (const void *)fft_any_kernel<kGenNoise>,
                         (const void *)fft_any_kernel<kPassY>,     (const void *)fft_any_kernel<kPassX>,
                         (const void *)fft_any_kernel<kFwdX>,      (const void *)fft_any_kernel<kPowZ>};
    for (const void *k : any) {
        hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds);
        if (e != hipSuccess) return rc = tt::hip_check(e, "hipFuncSetAttribute(max dynamic LDS)");
    }
#define FIXED(M)                                                                                              \
    (const void *)fft_pass_kernel<M, 128>, (const void *)fft_pass_kernel<M, 192>,                             \
        (const void *)fft_pass_kernel<M, 256>, (const void *)fft_pass_kernel<M, 384>,                         \
        (const void *)fft_pass_kernel<M, 512>, (const void *)fft_pass_kernel<M, 1024>
    const void *fixed[] = {FIXED(kGenNative), FIXED(kGenNoise), FIXED(kPassY),
                           FIXED(kPassX),     FIXED(kFwdX),     FIXED(kPowZ)};
#undef FIXED
    const int want = (int)(smem_fixed(1024) + 2 * kMaxBins * sizeof(double));
    for (const void *k : fixed) {
        hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, want);
        if (e != hipSuccess) return rc = tt::hip_check(e, "hipFuncSetAttribute(max dynamic LDS)");
    }
    return rc = TT_OK;
}

// one pass along axis ax (0 x, 1 y, 2 z) of the plan: the fixed-length kernel
// for 128, 192, 256, 384, 512 and 1024, the one for any length otherwise.
// extra: LDS behind the FFT's (power-spectrum bins)
template <int MODE>
void launch_pass(tt_fft_plan plan, int ax, hipStream_t st, PassArgs a, size_t extra = 0) {
    const int n = plan->ax[ax].n;
    a.ap = plan->ax[ax];
    a.tw = plan->tw[ax];
    constexpr bool kRows = MODE == kPassX || MODE == kFwdX;
    const int64_t count = kRows ? (int64_t)plan->ny * plan->nz : (int64_t)plan->nxh * (MODE == kPassY ? plan->nz : plan->ny);
    if (!fixed_length(n)) {
        a.lb = pencils_any(n, count, extra);
        const tt::Blocks b = tt::spread(tt::ceil_div(count, (int64_t)1 << a.lb), kAnyThreads);
        hipLaunchKernelGGL(fft_any_kernel<MODE>, dim3(b.x, b.y), dim3(kAnyThreads), smem_any(n, a.lb) + extra, st, a);
        return;
    }
    const int64_t B = kBatch / n;
    const dim3 grid = kRows ? dim3((unsigned)tt::ceil_div(count, B))
                    : MODE == kPowZ
                        ? dim3((unsigned)std::min<int64_t>(tt::ceil_div(count, B), kPowBlocks))
                        : dim3((unsigned)tt::ceil_div(plan->nxh, B), (unsigned)(MODE == kPassY ? plan->nz : plan->ny));
    const size_t sm = smem_fixed(n) + extra;
    switch (n) {
        case 128: hipLaunchKernelGGL((fft_pass_kernel<MODE, 128>), grid, dim3(kThreads), sm, st, a); break;
        case 192: hipLaunchKernelGGL((fft_pass_kernel<MODE, 192>), grid, dim3(kThreads), sm, st, a); break;
        case 256: hipLaunchKernelGGL((fft_pass_kernel<MODE, 256>), grid, dim3(kThreads), sm, st, a); break;
        case 384: hipLaunchKernelGGL((fft_pass_kernel<MODE, 384>), grid, dim3(kThreads), sm, st, a); break;
        case 512: hipLaunchKernelGGL((fft_pass_kernel<MODE, 512>), grid, dim3(kThreads), sm, st, a); break;
        default: hipLaunchKernelGGL((fft_pass_kernel<MODE, 1024>), grid, dim3(kThreads), sm, st, a); break;
    }
}

int run_passes(tt_fft_plan plan, PassArgs a, bool native, void *workspace, float *out, double *sumsq,
               hipStream_t st) {
    if (int rc = enable_lds()) return rc;
    a.nx = plan->nx;
    a.ny = plan->ny;
    a.nz = plan->nz;
    a.nxh = plan->nxh;
    a.spec = static_cast<float2 *>(workspace);
    a.out = out;
    a.sumsq = sumsq;
    a.scale = (float)(1.0 / ((double)plan->nx * plan->ny * plan->nz));
    if (native)
        launch_pass<kGenNative>(plan, 2, st, a);
    else
        launch_pass<kGenNoise>(plan, 2, st, a);
    TT_LAUNCH_CHECK("field pass Z launch");
    launch_pass<kPassY>(plan, 1, st, a);
    TT_LAUNCH_CHECK("field pass Y launch");
    launch_pass<kPassX>(plan, 0, st, a);
    TT_LAUNCH_CHECK("field pass X launch");
    return TT_OK;
}

}  // namespace

extern "C" int tt_field_generate(tt_fft_plan plan, const tt_spectrum *spec, void *workspace, float *out,
                                 double *sumsq, void *stream) {
    TT_REQUIRE(plan && spec && workspace && out, "tt_field_generate: null pointer");
    TT_REQUIRE(spec->aniso > 0, "tt_field_generate: aniso must be > 0");
    TT_REQUIRE(spec->amp >= 0, "tt_field_generate: amp must be >= 0");
    PassArgs a{};
    a.aniso = spec->aniso;
    a.kmin = spec->kmin;
    a.kmax = spec->kmax;
    a.half_beta = (float)(0.5 * spec->beta);
    a.sqrt_amp = (float)sqrt(spec->amp);
    a.key0 = (uint32_t)spec->seed;
    a.key1 = (uint32_t)(spec->seed >> 32);
    return run_passes(plan, a, true, workspace, out, sumsq, tt::as_stream(stream));
}

extern "C" int tt_field_from_noise(tt_fft_plan plan, const float *wr, const float *wi, const float *sqrt_psd,
                                   void *workspace, float *out, double *sumsq, void *stream) {
    TT_REQUIRE(plan && wr && wi && sqrt_psd && workspace && out, "tt_field_from_noise: null pointer");
    PassArgs a{};
    a.wr = wr;
    a.wi = wi;
    a.sp = sqrt_psd;
    return run_passes(plan, a, false, workspace, out, sumsq, tt::as_stream(stream));
}

extern "C" int tt_power_spectrum(tt_fft_plan plan, const float *field, int32_t mode, int32_t nbins, double dx,
                                 double bin_w, void *workspace, double *sums, double *counts, void *stream) {
    TT_REQUIRE(plan && field && workspace && sums && counts, "tt_power_spectrum: null pointer");
    TT_REQUIRE(mode == 0 || mode == 1, "tt_power_spectrum: mode must be 0 (spectrum_3D_scalar) or 1 (compute3Dspectrum)");
    TT_REQUIRE(nbins >= 1 && nbins <= kMaxBins, "tt_power_spectrum: nbins must be in [1, %d]", kMaxBins);
    TT_REQUIRE(dx > 0, "tt_power_spectrum: dx must be > 0");
    TT_REQUIRE(mode == 1 || bin_w > 0, "tt_power_spectrum: bin_w must be > 0");
    if (int rc = enable_lds()) return rc;
    hipStream_t st = tt::as_stream(stream);
    PassArgs a{};
    a.nx = plan->nx;
    a.ny = plan->ny;
    a.nz = plan->nz;
    a.nxh = plan->nxh;
    a.spec = static_cast<float2 *>(workspace);
    a.in = field;
    a.mode = mode;
    a.nbins = nbins;
    // numpy fftfreq(M, d): integer index times 1.0 / (M * d)
    a.fx_step = 1.0 / ((double)plan->nx * dx);
    a.fy_step = 1.0 / ((double)plan->ny * dx);
    a.fz_step = 1.0 / ((double)plan->nz * dx);
    a.bin_w = bin_w;
    a.inv_bin_w = mode == 0 ? 1.0 / bin_w : 0.0;
    const double nt = (double)plan->nx * plan->ny * plan->nz;
    a.pscale = mode == 0 ? 1.0 : 1.0 / (nt * nt);
    a.hsum = sums;
    a.hcnt = counts;
    launch_pass<kFwdX>(plan, 0, st, a);  // real rows -> half spectrum
    TT_LAUNCH_CHECK("power spectrum pass X launch");
    launch_pass<kPassY>(plan, 1, st, a);
    TT_LAUNCH_CHECK("power spectrum pass Y launch");
    // pass Z with |F|^2 binning (sums and counts are ADDED to)
    launch_pass<kPowZ>(plan, 2, st, a, 2 * (size_t)nbins * sizeof(double));
    TT_LAUNCH_CHECK("power spectrum pass Z launch");
    return TT_OK;
}
