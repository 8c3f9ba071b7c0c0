// convolve.hip -- auralization: convolution of impulse-response tracks with
// a sound signal (RecorderTrack::Process, src/Recorder.cpp:145-243).
//
// The reference transforms the zero-padded track a and signal b (both of
// length M + N + 1) with FFTW, multiplies the spectra, scales by 1 / (M + N + 1)
// and transforms back; with a second track (keyframe interpolation) it adds
// the convolution of that track with the signal faded in to the convolution
// of the first with the signal faded out.  Here the transforms have a
// power-of-two length L >= M + N + 1 (more zero padding leaves the linear
// convolution unchanged), and both products are summed in the frequency
// domain, so one inverse transform serves both terms.
//
// Up to 2^22 samples (95 s) the transforms are the kernels below, in
// binary64; longer ones are batched hipFFT real transforms.  What bounded a
// call was the library's plan, made and dropped with its code objects on every
// call: 24 of 26 ms for 3 s of response and 10 s of faded sound, whose kernels
// took 0.3 ms.
#include <hip/hip_runtime.h>
#include <hipfft/hipfft.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "ear_internal.hpp"

namespace ear {
namespace {

// C[k] = (A0[k] B0[k] + A1[k] B1[k]) * scale over nc bins; terms = 1 or 2
__global__ void k_spectra_mul(const float2* __restrict__ X, uint32_t nc, uint32_t terms, float scale,
                              float2* __restrict__ C) {
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < nc; k += gridDim.x * blockDim.x) {
        float re = 0.0f, im = 0.0f;
        for (uint32_t t = 0; t < terms; ++t) {
            const float2 a = X[(size_t)t * nc + k];                // track t
            const float2 b = X[((size_t)terms + t) * nc + k];      // signal t
            re += a.x * b.x - a.y * b.y;
            im += a.x * b.y + a.y * b.x;
        }
        C[k] = make_float2(re * scale, im * scale);
    }
}

// ---------------------------------------------------------------------------
// The convolution.  A track and its signal are the real and
// imaginary parts of one sequence z of L = N1 N2 values.  Index n = n1 N2 + n2:
//   k_conv_peaks    the operands' largest samples (see Level)
//   k_conv_columns  the N1-point transforms down the columns n2, times
//                   e^(-2 pi i k1 n2 / L); reads the real inputs, writes z
//   k_conv_rows     the N2-point transforms along the rows k1 (frequency
//                   k1 + N1 k2 at [k1][k2]), the spectra's product, and the
//                   inverse transforms of the rows: a workgroup holds row k1
//                   and row N1 - k1, because frequency -k, which separates the
//                   track's spectrum from the signal's, lies there
//   k_conv_out      the inverse transforms of the columns; writes the samples
// so z crosses memory twice each way and no reordering pass is needed.
// binary64: the vector unit's rate is close to binary32's, the sequence
// (L = 2^20: 16 MB) stays in the caches, and the result is then the exact
// convolution rounded once (6e-8 of the largest sample, 2.7e-7 with binary32
// transforms).  4096 values a workgroup (96 KB of LDS with the roots, so one
// workgroup a CU; 16 registers' worth per thread) whatever the shape.  3 s of
// response and 10 s of faded sound: 0.80 ms a call, with and without the pass
// over the operands' sizes; the copies to and from the host are most of it.
// ---------------------------------------------------------------------------
constexpr int kConvThreads = 256;
constexpr int kConvValues = 4096;
constexpr int kConvMinLog = 12, kConvMaxLog = 22;  // N1 and N2 are 2^6 .. 2^11

struct ConvTerm {
    const float* track;
    const float* signal;
    uint32_t n_track, n_signal;
};

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// The rounding of a transform is relative to the largest of what it holds, so a
// track and its signal go into one sequence each divided by the power of two
// 2^e that brings its largest sample into [1/2, 1) (exact); the product is
// scaled back before the terms are summed.  Without it a response 1e-12 of its
// sound kept 3 digits.  A term with nothing in its track or signal adds nothing.
struct Level {
    uint32_t bits;  // of the largest |sample|; above infinity's: a NaN
    __device__ __forceinline__ bool silent() const { return bits == 0; }
    __device__ __forceinline__ bool finite() const { return bits < 0x7F800000u; }
    __device__ __forceinline__ int exponent() const {
        if (silent() || !finite()) return 0;
        return bits >> 23 ? (int)(bits >> 23) - 126 : (32 - __clz((int)bits)) - 149;
    }
};
constexpr int kPeakBlocks = 64;  // partial maxima of an operand: one a lane

// block (b, 2 term + {0 track, 1 signal}): the largest |sample| of every
// kPeakBlocks-th run of the operand
__global__ void __launch_bounds__(kConvThreads) k_conv_peaks(ConvTerm t0, ConvTerm t1, uint32_t* __restrict__ peaks) {
    const ConvTerm t = blockIdx.y >> 1 ? t1 : t0;
    const float* x = blockIdx.y & 1u ? t.signal : t.track;
    const uint32_t n = blockIdx.y & 1u ? t.n_signal : t.n_track;
    uint32_t m = 0;
    for (uint32_t i = blockIdx.x * kConvThreads + threadIdx.x; i < n; i += kPeakBlocks * kConvThreads)
        m = max(m, __float_as_uint(x[i]) & 0x7FFFFFFFu);
    for (int o = 32; o; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o));
    __shared__ uint32_t wave[kConvThreads / 64];
    if ((threadIdx.x & 63u) == 0) wave[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kConvThreads / 64; ++w) m = max(m, wave[w]);
        peaks[blockIdx.y * kPeakBlocks + blockIdx.x] = m;
    }
}

// the whole wave calls it
__device__ __forceinline__ Level level_of(const uint32_t* peaks, uint32_t operand) {
    uint32_t m = peaks[operand * kPeakBlocks + (threadIdx.x & 63u)];
    for (int o = 32; o; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o));
    return Level{(uint32_t)__builtin_amdgcn_readfirstlane((int)m)};
}
// (silence beside a NaN or an infinity is carried on: it makes NaNs)
__device__ __forceinline__ bool nothing(Level a, Level b) {
    return (a.silent() && b.finite()) || (b.silent() && a.finite());
}

// e^(2 pi i num / 2^lg); num / 2^lg is exact
__device__ __forceinline__ double2 unit_root(double num, int lg) {
    double s, c;
    sincospi(ldexp(num, 1 - lg), &s, &c);
    return make_double2(c, s);
}

// nb transforms of 2^lg values each (nb 2^lg <= kConvValues) at x[b 2^lg ..] in
// LDS, in order: Stockham's radix-4 passes (a radix-2 one last for odd lg),
// every value read before any is written.  tw: e^(-2 pi i j / 2^lg).  INV:
// the conjugate transform, unscaled.  The whole workgroup calls it.
template <bool INV>
__device__ void lds_fft(double2* x, const double2* tw, int lg, int nb) {
    const int N = 1 << lg, quarter = N >> 2;
    for (int ls = 0; ls + 2 <= lg; ls += 2) {
        const int total = nb * quarter;
        double2 v[4][4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int idx = (int)threadIdx.x + j * kConvThreads;
            if (idx < total) {
                const double2* b = x + ((idx >> (lg - 2)) << lg) + (idx & (quarter - 1));
#pragma unroll
                for (int k = 0; k < 4; ++k) v[j][k] = b[k * quarter];
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int idx = (int)threadIdx.x + j * kConvThreads;
            if (idx < total) {
                const int t = idx & (quarter - 1), q = t & ((1 << ls) - 1), ps = t - q;  // ps = p << ls
                double2 w1 = tw[ps], w2 = tw[2 * ps], w3 = tw[3 * ps];
                if (INV) {
                    w1.y = -w1.y;
                    w2.y = -w2.y;
                    w3.y = -w3.y;
                }
                const double2 a = v[j][0], b = v[j][1], c = v[j][2], d = v[j][3];
                const double2 apc = make_double2(a.x + c.x, a.y + c.y), amc = make_double2(a.x - c.x, a.y - c.y);
                const double2 bpd = make_double2(b.x + d.x, b.y + d.y);
                // i (b - d), its sign by direction
                const double2 jb = INV ? make_double2(b.y - d.y, d.x - b.x) : make_double2(d.y - b.y, b.x - d.x);
                double2* o = x + ((idx >> (lg - 2)) << lg) + q + 4 * ps;
                o[0] = make_double2(apc.x + bpd.x, apc.y + bpd.y);
                o[1 << ls] = cmul(w1, make_double2(amc.x - jb.x, amc.y - jb.y));
                o[2 << ls] = cmul(w2, make_double2(apc.x - bpd.x, apc.y - bpd.y));
                o[3 << ls] = cmul(w3, make_double2(amc.x + jb.x, amc.y + jb.y));
            }
        }
        __syncthreads();
    }
    if (lg & 1) {
        const int half = N >> 1;
        for (int idx = (int)threadIdx.x; idx < nb * half; idx += kConvThreads) {
            double2* b = x + ((idx >> (lg - 1)) << lg) + (idx & (half - 1));
            const double2 u = b[0], w = b[half];
            b[0] = make_double2(u.x + w.x, u.y + w.y);
            b[half] = make_double2(u.x - w.x, u.y - w.y);
        }
        __syncthreads();
    }
}

__device__ __forceinline__ void fill_roots(double2* tw, int lg) {
    for (int j = (int)threadIdx.x; j < (1 << lg); j += kConvThreads) tw[j] = unit_root(-(double)j, lg);
}

// block: kConvValues >> lg1 columns of term blockIdx.y
__global__ void __launch_bounds__(kConvThreads) k_conv_columns(ConvTerm t0, ConvTerm t1, int lg1, int lg2,
                                                               const uint32_t* __restrict__ peaks,
                                                               double2* __restrict__ z) {
    __shared__ double2 x[kConvValues];
    __shared__ double2 tw[1 << (kConvMaxLog / 2)];
    const ConvTerm t = blockIdx.y ? t1 : t0;
    const int lc = kConvMinLog - lg1, C = 1 << lc;  // kConvValues = 2^kConvMinLog
    const uint32_t c0 = blockIdx.x << lc;
    const Level la = level_of(peaks, 2 * blockIdx.y), lb = level_of(peaks, 2 * blockIdx.y + 1);
    if (nothing(la, lb)) return;  // k_conv_rows leaves the term out
    const double sa = ldexp(1.0, -la.exponent()), sb = ldexp(1.0, -lb.exponent());
    fill_roots(tw, lg1);
    for (int e = (int)threadIdx.x; e < kConvValues; e += kConvThreads) {
        const uint32_t n1 = (uint32_t)e >> lc, c = (uint32_t)e & (C - 1), n = (n1 << lg2) + c0 + c;
        x[(c << lg1) + n1] = make_double2(n < t.n_track ? (double)t.track[n] * sa : 0.0,
                                          n < t.n_signal ? (double)t.signal[n] * sb : 0.0);
    }
    __syncthreads();
    lds_fft<false>(x, tw, lg1, C);
    double2* out = z + ((size_t)blockIdx.y << (lg1 + lg2));
    for (int e = (int)threadIdx.x; e < kConvValues; e += kConvThreads) {
        const uint32_t k1 = (uint32_t)e >> lc, c = (uint32_t)e & (C - 1);
        const double2 w = unit_root(-((double)k1 * (double)(c0 + c)), lg1 + lg2);
        out[((size_t)k1 << lg2) + c0 + c] = cmul(x[(c << lg1) + k1], w);
    }
}

// block k1 = 0 .. N1 / 2: rows k1 and N1 - k1 of every term; the product's
// rows replace the first term's
__global__ void __launch_bounds__(kConvThreads) k_conv_rows(int terms, int lg1, int lg2,
                                                            const uint32_t* __restrict__ peaks,
                                                            double2* __restrict__ z) {
    __shared__ double2 x[kConvValues];
    __shared__ double2 tw[1 << (kConvMaxLog / 2)];
    constexpr int kPer = kConvValues / 2 / kConvThreads;  // frequencies per thread and row
    const int N1 = 1 << lg1, N2 = 1 << lg2;
    const int ra = (int)blockIdx.x, rb = (N1 - ra) & (N1 - 1);
    fill_roots(tw, lg2);
    double2 acc[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) acc[j] = make_double2(0.0, 0.0);
    // frequency -k of [ra][k2] is [rb][mirror(k2)]
    auto mirror = [&](int k2) { return ra == 0 ? (N2 - k2) & (N2 - 1) : N2 - 1 - k2; };
    for (int t = 0; t < terms; ++t) {
        const Level la = level_of(peaks, 2 * t), lb = level_of(peaks, 2 * t + 1);
        if (nothing(la, lb)) continue;
        const double back = ldexp(1.0, la.exponent() + lb.exponent());
        const double2* in = z + ((size_t)t << (lg1 + lg2));
        for (int e = (int)threadIdx.x; e < 2 * N2; e += kConvThreads)
            x[e] = in[((size_t)(e < N2 ? ra : rb) << lg2) + (e & (N2 - 1))];
        __syncthreads();
        lds_fft<false>(x, tw, lg2, 2);
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const int k2 = (int)threadIdx.x + j * kConvThreads;
            if (k2 < N2) {
                // z = a + i b of real a, b: A = (Z(k) + Z(-k)*) / 2, B = (Z(k) - Z(-k)*) / 2i
                const double2 u = x[k2], v = x[N2 + mirror(k2)];
                const double2 A = make_double2(0.5 * (u.x + v.x), 0.5 * (u.y - v.y));
                const double2 B = make_double2(0.5 * (u.y + v.y), 0.5 * (v.x - u.x));
                const double2 P = cmul(A, B);
                acc[j].x += P.x * back;
                acc[j].y += P.y * back;
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int k2 = (int)threadIdx.x + j * kConvThreads;
        if (k2 < N2) {
            x[k2] = acc[j];
            x[N2 + mirror(k2)] = make_double2(acc[j].x, -acc[j].y);
        }
    }
    __syncthreads();
    lds_fft<true>(x, tw, lg2, 2);
    for (int e = (int)threadIdx.x; e < (ra == rb ? N2 : 2 * N2); e += kConvThreads) {
        const int r = e < N2 ? ra : rb, n2 = e & (N2 - 1);
        z[((size_t)r << lg2) + n2] = cmul(x[e], unit_root((double)r * (double)n2, lg1 + lg2));
    }
}

__global__ void __launch_bounds__(kConvThreads) k_conv_out(int lg1, int lg2, const double2* __restrict__ z,
                                                           uint32_t n_out, float* __restrict__ out) {
    __shared__ double2 x[kConvValues];
    __shared__ double2 tw[1 << (kConvMaxLog / 2)];
    const int lc = kConvMinLog - lg1, C = 1 << lc;
    const uint32_t c0 = blockIdx.x << lc;
    fill_roots(tw, lg1);
    for (int e = (int)threadIdx.x; e < kConvValues; e += kConvThreads) {
        const uint32_t k1 = (uint32_t)e >> lc, c = (uint32_t)e & (C - 1);
        x[(c << lg1) + k1] = z[((size_t)k1 << lg2) + c0 + c];
    }
    __syncthreads();
    lds_fft<true>(x, tw, lg1, C);
    const double scale = ldexp(1.0, -(lg1 + lg2));
    for (int e = (int)threadIdx.x; e < kConvValues; e += kConvThreads) {
        const uint32_t n1 = (uint32_t)e >> lc, c = (uint32_t)e & (C - 1), n = (n1 << lg2) + c0 + c;
        if (n < n_out) out[n] = (float)(x[(c << lg1) + n1].x * scale);
    }
}

ear_status convolve_short(Ctx* c, const float* const* tracks, const uint32_t* n_track, const float* const* signals,
                          uint32_t terms, uint32_t n_sig, float* out, uint32_t n_out, int lg) {
    const int lg2 = lg / 2, lg1 = lg - lg2;
    hipStream_t st = c->stream;
    DevBuf in(c), z(c), res(c), peaks(c);
    size_t n_in = (size_t)terms * n_sig;
    for (uint32_t t = 0; t < terms; ++t) n_in += n_track[t];
    TRY(in.alloc(n_in * sizeof(float)));
    TRY(z.alloc(((size_t)terms << lg) * sizeof(double2)));
    TRY(res.alloc((size_t)n_out * sizeof(float)));
    TRY(peaks.alloc(2 * terms * kPeakBlocks * sizeof(uint32_t)));
    ConvTerm term[2] = {};
    float* p = in.as<float>();
    for (uint32_t t = 0; t < terms; ++t) {
        term[t] = ConvTerm{p, p + n_track[t], n_track[t], n_sig};
        EAR_HIP_TRY(c, hipMemcpyAsync(p, tracks[t], (size_t)n_track[t] * 4, hipMemcpyHostToDevice, st));
        EAR_HIP_TRY(c, hipMemcpyAsync(p + n_track[t], signals[t], (size_t)n_sig * 4, hipMemcpyHostToDevice, st));
        p += n_track[t] + n_sig;
    }
    const uint32_t cols = (1u << lg2) >> (kConvMinLog - lg1);  // workgroups of columns
    k_conv_peaks<<<dim3(kPeakBlocks, 2 * terms), kConvThreads, 0, st>>>(term[0], term[1], peaks.as<uint32_t>());
    k_conv_columns<<<dim3(cols, terms), kConvThreads, 0, st>>>(term[0], term[1], lg1, lg2, peaks.as<uint32_t>(),
                                                               z.as<double2>());
    k_conv_rows<<<(1u << lg1) / 2 + 1, kConvThreads, 0, st>>>((int)terms, lg1, lg2, peaks.as<uint32_t>(),
                                                              z.as<double2>());
    k_conv_out<<<cols, kConvThreads, 0, st>>>(lg1, lg2, z.as<double2>(), n_out, res.as<float>());
    EAR_HIP_TRY(c, hipGetLastError());
    EAR_HIP_TRY(c, hipMemcpyAsync(out, res.p, (size_t)n_out * 4, hipMemcpyDeviceToHost, st));
    EAR_HIP_TRY(c, hipStreamSynchronize(st));
    return EAR_OK;
}

struct Plan {
    hipfftHandle h = 0;
    ~Plan() {
        if (h) hipfftDestroy(h);
    }
};

ear_status fft_status(Ctx* c, hipfftResult r, const char* what) {
    if (r == HIPFFT_SUCCESS) return EAR_OK;
    c->last_error = std::string(what) + " failed (hipFFT error " + std::to_string((int)r) + ")";
    return r == HIPFFT_ALLOC_FAILED ? EAR_ERR_OUT_OF_MEMORY : EAR_ERR_HIP;
}

}  // namespace

ear_status run_convolve(Ctx* c, const float* const* tracks, const uint32_t* n_track, const float* const* signals,
                        uint32_t terms, uint32_t n_sig, float* out, uint32_t n_out) {
    uint64_t need = n_out;
    uint32_t L = 1;
    while (L < need) L <<= 1;
    int lg = kConvMinLog;
    while (lg < 31 && (1u << lg) < L) ++lg;
    if (lg <= kConvMaxLog) return convolve_short(c, tracks, n_track, signals, terms, n_sig, out, n_out, lg);
    const uint32_t nc = L / 2 + 1;
    hipStream_t st = c->stream;
    DevBuf real(c), spec(c), prod(c);
    // inputs: tracks then signals, each zero-padded to L reals
    TRY(real.alloc((size_t)2 * terms * L * sizeof(float)));
    TRY(spec.alloc((size_t)2 * terms * nc * sizeof(float2)));
    TRY(prod.alloc((size_t)nc * sizeof(float2)));
    EAR_HIP_TRY(c, hipMemsetAsync(real.p, 0, real.n, st));
    for (uint32_t t = 0; t < terms; ++t) {
        EAR_HIP_TRY(c, hipMemcpyAsync(real.as<float>() + (size_t)t * L, tracks[t], (size_t)n_track[t] * 4,
                                      hipMemcpyHostToDevice, st));
        EAR_HIP_TRY(c, hipMemcpyAsync(real.as<float>() + (size_t)(terms + t) * L, signals[t], (size_t)n_sig * 4,
                                      hipMemcpyHostToDevice, st));
    }
    Plan fwd, inv;
    int n = (int)L;
    int inembed = (int)L, onembed = (int)nc;
    TRY(fft_status(c, hipfftPlanMany(&fwd.h, 1, &n, &inembed, 1, (int)L, &onembed, 1, (int)nc, HIPFFT_R2C,
                                     (int)(2 * terms)),
                   "hipfftPlanMany (forward)"));
    TRY(fft_status(c, hipfftPlan1d(&inv.h, n, HIPFFT_C2R, 1), "hipfftPlan1d (inverse)"));
    TRY(fft_status(c, hipfftSetStream(fwd.h, st), "hipfftSetStream"));
    TRY(fft_status(c, hipfftSetStream(inv.h, st), "hipfftSetStream"));
    TRY(fft_status(c, hipfftExecR2C(fwd.h, real.as<hipfftReal>(), spec.as<hipfftComplex>()), "forward FFT"));
    k_spectra_mul<<<std::min<uint32_t>((nc + 255) / 256, 4096), 256, 0, st>>>(spec.as<float2>(), nc, terms,
                                                                            1.0f / (float)L, prod.as<float2>());
    EAR_HIP_TRY(c, hipGetLastError());
    TRY(fft_status(c, hipfftExecC2R(inv.h, prod.as<hipfftComplex>(), real.as<hipfftReal>()), "inverse FFT"));
    EAR_HIP_TRY(c, hipMemcpyAsync(out, real.p, (size_t)n_out * 4, hipMemcpyDeviceToHost, st));
    EAR_HIP_TRY(c, hipStreamSynchronize(st));
    return EAR_OK;
}

}  // namespace ear
