// Spectral analysis of recorded traces: the transforms of the reference's
// analysis.spectrum (phonomena/simulation/analysis.py:44-96), which takes
// |fft(u * hann, norm="ortho")| of a time trace, or |fft2| of an (x, t)
// slice, and keeps the first N//2 frequencies.
//
// pf_dft: a batch of 1-D discrete Fourier transforms along the contiguous
// axis, in FP64, for the first nf frequencies:
//     out[b, k] = scale * sum_t (in[b, t] * w[t]) e^{-2 pi i k t / n}
// in O(n log n) per trace, for any n:
//
//  * n a power of two up to 8192: an FFT of length M = n.
//  * any other n (up to 2^23): Bluestein's chirp-z form.  With c_m = e^{-pi i m^2 / n},
//    k t = (k^2 + t^2 - (k - t)^2) / 2 turns the transform into
//        X_k = c_k sum_t (a_t c_t) conj(c_{k-t}),
//    a convolution, evaluated as a circular one of power-of-two length
//    M >= n + nf - 1 (the lags -(n-1) .. nf-1 stay apart, so the first half
//    of the frequencies takes a shorter M than all of them) through two
//    FFTs and the transform of the wrapped chirp conj(c).  m^2 is reduced
//    mod 2n in integers, so no angle loses precision however long the trace.
//
// Every FFT runs in LDS in radix-8 passes (a last one of 4 or 2), a
// butterfly in a thread's registers: decimation in frequency forward
// (natural-order input, digit-reversed output) and decimation in time with
// conjugate twiddles back, so the convolution reorders nothing; a plain
// transform reads its output through the digit reversal.  Elements are
// padded by one in eight: the last passes' stride of 8 values would meet in
// one bank.  Against radix-2 passes this is a third of the LDS traffic and
// barriers.  M <= 8192 (144 KB): one block per trace does the whole
// transform in LDS.  Longer: M = M1 * M2 with t = M2 t1 + t2,
// k = k1 + M1 k2 (the four-step split), in three launches over a scratch of
// M values per trace (rows in the digit-reversed order of k1 throughout):
//   1. length-M1 FFTs over t1 (several t2 columns per block, read as
//      contiguous runs), times e^{-2 pi i t2 k1 / M}, stored as [k1][t2];
//   2. per row k1: length-M2 FFT over t2 (now X at k1 + M1 k2), times the
//      chirp transform (kept in the same order), the inverse length-M2 FFT,
//      times e^{+2 pi i k1 t2 / M};
//   3. inverse length-M1 FFTs over k1, times c_k * scale / M, the first nf
//      frequencies stored.
// The tables (twiddles, chirp) are made on the device from exact fractions
// of a turn; e^{-2 pi i m / M} for the four-step factor is the product of two
// table entries (m = a M2 + b).  Every product is plain FP64 arithmetic;
// the results differ from numpy's FFT by rounding only.
//
// Measured, the whole call with Hann window and the first half of the
// frequencies (before: radix-2 passes, M >= 2n - 1, tables made on the host
// on each call, a device allocation per array, pageable copies): 1024 traces
// of 5000 values 3.0 ms (15.8), 64 of 50,000 2.3 (12.0), 8 of 400,000 2.5
// (16.1), one of 5000 0.10 (0.57).  Of the first, 6.4 with pageable copies,
// the kernels are 0.4 and the two staged copies (pf_stage.hpp) the rest.  The
// error against 64 bits went from 9e-16 to 6e-16 (relative 2-norm).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "../../include/phonofdtd.h"
#include "pf_runtime.hpp"
#include "pf_stage.hpp"

using namespace pf;

namespace {

constexpr int FFT_LG_SMALL = 13;  // one block, whole transform in LDS: M <= 8192
constexpr int FFT_LG_TILE = 12;   // four-step blocks hold 4096 values
constexpr int FFT_LG_MAX = 24;    // M <= 2^24: n <= 2^23 for Bluestein
constexpr int FFT_TILE_THREADS = 256;

constexpr int padded(int n) { return n + n / 8; }
__device__ __forceinline__ int pad(int i) { return i + (i >> 3); }

__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cmulc(double2 a, double2 b) {  // a * conj(b)
    return make_double2(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y);
}
// a * -i (forward), a * +i (inverse)
template <bool INV> __device__ __forceinline__ double2 mul_i(double2 a) {
    return INV ? make_double2(-a.y, a.x) : make_double2(a.y, -a.x);
}

// DFT of v[0 .. 2^B) in place, natural order in and out.
template <int B, bool INV> __device__ __forceinline__ void dft(double2* v) {
    if constexpr (B == 1) {
        const double2 a = v[0];
        v[0] = cadd(a, v[1]);
        v[1] = csub(a, v[1]);
    } else if constexpr (B == 2) {
        const double2 a = cadd(v[0], v[2]), b = csub(v[0], v[2]), c = cadd(v[1], v[3]),
                      d = mul_i<INV>(csub(v[1], v[3]));
        v[0] = cadd(a, c);
        v[1] = cadd(b, d);
        v[2] = csub(a, c);
        v[3] = csub(b, d);
    } else {
        constexpr double h = 0.70710678118654752440;  // sqrt(1/2)
        double2 e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
        dft<2, INV>(e);
        dft<2, INV>(o);
        // times e^{-+pi i k / 4}
        const double2 t1 = mul_i<INV>(o[1]), t3 = mul_i<INV>(o[3]);
        o[1] = make_double2(h * (o[1].x + t1.x), h * (o[1].y + t1.y));
        o[2] = mul_i<INV>(o[2]);
        o[3] = make_double2(h * (t3.x - o[3].x), h * (t3.y - o[3].y));
#pragma unroll
        for (int k = 0; k < 4; k++) {
            v[k] = cadd(e[k], o[k]);
            v[k + 4] = csub(e[k], o[k]);
        }
    }
}

// One radix-2^B pass over N values in LDS, blocks of 2^l.  tw holds
// e^{-2 pi i j / 2^tlg} for the first half turn.  Ends with a barrier.
template <int B, bool INV>
__device__ __forceinline__ void fft_pass(double2* s, int N, int l, const double2* __restrict__ tw, int tlg) {
    constexpr int R = 1 << B;
    const int lh = l - B, h = 1 << lh;
    for (int q = threadIdx.x; q < N >> B; q += blockDim.x) {
        const int j = q & (h - 1), base = ((q >> lh) << l) + j;
        double2 v[R], w[R];
#pragma unroll
        for (int m = 0; m < R; m++) v[m] = s[pad(base + (m << lh))];
        w[1] = tw[j << (tlg - l)];
        if constexpr (B >= 2) {
            w[2] = tw[(2 * j) << (tlg - l)];
            w[3] = cmul(w[1], w[2]);
        }
        if constexpr (B == 3) {
            w[4] = tw[(4 * j) << (tlg - l)];
            w[5] = cmul(w[1], w[4]);
            w[6] = cmul(w[2], w[4]);
            w[7] = cmul(w[3], w[4]);
        }
        if constexpr (INV) {
#pragma unroll
            for (int m = 1; m < R; m++) v[m] = cmulc(v[m], w[m]);
        }
        dft<B, INV>(v);
        if constexpr (!INV) {
#pragma unroll
            for (int m = 1; m < R; m++) v[m] = cmul(v[m], w[m]);
        }
#pragma unroll
        for (int m = 0; m < R; m++) s[pad(base + (m << lh))] = v[m];
    }
    __syncthreads();
}

// N / 2^lg transforms of length 2^lg, each contiguous in s, in place:
// natural order to digit-reversed.  Begins and ends with a barrier.
__device__ void fft_fwd(double2* s, int N, int lg, const double2* __restrict__ tw, int tlg) {
    __syncthreads();
    int l = lg;
    for (; l >= 3; l -= 3) fft_pass<3, false>(s, N, l, tw, tlg);
    if (l == 2) fft_pass<2, false>(s, N, 2, tw, tlg);
    else if (l == 1) fft_pass<1, false>(s, N, 1, tw, tlg);
}
// Digit-reversed to natural order, without the 1 / 2^lg.
__device__ void fft_inv(double2* s, int N, int lg, const double2* __restrict__ tw, int tlg) {
    __syncthreads();
    int l = lg % 3;
    if (l == 2) fft_pass<2, true>(s, N, 2, tw, tlg);
    else if (l == 1) fft_pass<1, true>(s, N, 1, tw, tlg);
    for (l += 3; l <= lg; l += 3) fft_pass<3, true>(s, N, l, tw, tlg);
}
// Frequency at position p of a forward transform's output, and back.
__device__ __forceinline__ int freq_at(int p, int lg) {
    int k = 0, shift = 0;
    for (int l = lg; l > 0;) {
        const int b = l >= 3 ? 3 : l;
        l -= b;
        k |= ((p >> l) & ((1 << b) - 1)) << shift;
        shift += b;
    }
    return k;
}
__device__ __forceinline__ int pos_of(int k, int lg) {
    int p = 0;
    for (int l = lg; l > 0;) {
        const int b = l >= 3 ? 3 : l;
        l -= b;
        p |= (k & ((1 << b) - 1)) << l;
        k >>= b;
    }
    return p;
}

// A batch of traces: value t of trace b at re[(b n + t) step] (im alike, or
// null), times win[t] (or 1).
struct Traces {
    const double* re;
    const double* im;
    const double* win;
    long long n;
    int step;
};
// Its first nf frequencies: frequency k of trace b to re / im[(b nf + k) step].
struct Spectra {
    double* re;
    double* im;
    long long nf;
    int step;
    double scale;
};

// Input value t of trace b, times the chirp (when there is one), zero past n.
__device__ __forceinline__ double2 load_in(const Traces& in, long long b, const double2* __restrict__ chirp,
                                           long long t) {
    double2 v = make_double2(0.0, 0.0);
    if (t < in.n) {
        const long long a = (b * in.n + t) * in.step;
        v.x = in.re[a];
        v.y = in.im ? in.im[a] : 0.0;
        if (in.win) {
            v.x = v.x * in.win[t];
            v.y = v.y * in.win[t];
        }
        if (chirp) v = cmul(v, chirp[t]);
    }
    return v;
}
// Value t of the wrapped conj chirp of length M: lags 0 .. nf-1 from the
// front, -(n-1) .. -1 from the back.
__device__ __forceinline__ double2 load_chirp(const double2* __restrict__ chirp, long long n, long long nf, long long M,
                                              long long t) {
    const long long m = t < nf ? t : M - t;
    if (t >= nf && m >= n) return make_double2(0.0, 0.0);
    return make_double2(chirp[m].x, -chirp[m].y);
}
__device__ __forceinline__ void store_out(const Spectra& o, long long b, long long k, double2 v) {
    const long long a = (b * o.nf + k) * o.step;
    o.re[a] = o.scale * v.x;
    o.im[a] = o.scale * v.y;
}

// e^{-2 pi i num / den}, num < 2^53 (an exact fraction of a turn).
__device__ __forceinline__ double2 unit(long long num, long long den) {
    double s, c;
    sincospi(2.0 * ((double)num / (double)den), &s, &c);
    return make_double2(c, -s);
}
// Tables: tw half a turn of 2^tlg; the chirp's n values (n = 0: none); for a
// four-step transform ta (1 << lg1, steps of 2^lg2 / 2^lg) and tb (1 << lg2).
struct Tables {
    double2 *tw, *chirp, *ta, *tb;
    long long n;
    int tlg, lg1, lg2;
};
__global__ __launch_bounds__(256) void k_fft_tables(Tables tb) {
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    if (t < (1ll << tb.tlg) / 2) tb.tw[t] = unit(t, 1ll << tb.tlg);
    if (t < tb.n)
        tb.chirp[t] = unit((long long)(((unsigned long long)t * (unsigned long long)t) % (2ull * tb.n)), 2 * tb.n);
    if (tb.ta) {
        if (t < (1ll << tb.lg1)) tb.ta[t] = unit(t << tb.lg2, 1ll << (tb.lg1 + tb.lg2));
        if (t < (1ll << tb.lg2)) tb.tb[t] = unit(t, 1ll << (tb.lg1 + tb.lg2));
    }
}

// e^{-2 pi i m / M}, m = a M2 + b, from the two tables.
__device__ __forceinline__ double2 twiddle_m(const double2* __restrict__ ta, const double2* __restrict__ tb,
                                             unsigned long long m, int lg2) {
    return cmul(ta[m >> lg2], tb[m & ((1ull << lg2) - 1)]);
}

// Whole transform of one trace (blockIdx.x) in LDS, M = 2^lg <= CAP.
//   bhat == nullptr, oc == nullptr: plain FFT (M = n), first nf values
//     times scale to out;
//   bhat != nullptr: Bluestein (chirp set), scale includes 1 / M;
//   oc != nullptr: forward FFT of the wrapped chirp, all M values stored to
//     oc in the transform's order.
template <int CAP>
__global__ __launch_bounds__(1024) void k_fft_small(Traces in, const double2* __restrict__ chirp,
                                                    const double2* __restrict__ bhat, int lg,
                                                    const double2* __restrict__ tw, Spectra out,
                                                    double2* __restrict__ oc) {
    __shared__ double2 s[padded(CAP)];
    const int M = 1 << lg;
    const long long b = blockIdx.x;
    for (int t = threadIdx.x; t < M; t += blockDim.x)
        s[pad(t)] = oc ? load_chirp(chirp, in.n, out.nf, M, t) : load_in(in, b, chirp, t);
    fft_fwd(s, M, lg, tw, lg);
    if (oc) {
        for (int t = threadIdx.x; t < M; t += blockDim.x) oc[t] = s[pad(t)];
        return;
    }
    if (bhat) {
        for (int t = threadIdx.x; t < M; t += blockDim.x) s[pad(t)] = cmul(s[pad(t)], bhat[t]);
        fft_inv(s, M, lg, tw, lg);
    }
    for (int k = threadIdx.x; k < out.nf; k += blockDim.x)
        store_out(out, b, k, bhat ? cmul(s[pad(k)], chirp[k]) : s[pad(pos_of(k, lg))]);
}

// Four-step, launch 1: grid (M2 / cb, traces); block x takes the cb
// columns t2 = cb x ... cb x + cb - 1 of trace blockIdx.y (of the wrapped
// chirp when `wrapped`).
__global__ __launch_bounds__(FFT_TILE_THREADS) void k_fft_cols(Traces in, const double2* __restrict__ chirp, bool wrapped,
                                                               long long nf, int lg1, int lg2, int lgcb,
                                                               const double2* __restrict__ tw,
                                                               const double2* __restrict__ ta,
                                                               const double2* __restrict__ tb,
                                                               double2* __restrict__ T) {
    __shared__ double2 s[padded(1 << FFT_LG_TILE)];
    const int M1 = 1 << lg1, cb = 1 << lgcb;
    const long long b = blockIdx.y, M = 1ll << (lg1 + lg2);
    const int c0 = blockIdx.x << lgcb;
    for (int q = threadIdx.x; q < cb * M1; q += blockDim.x) {
        const int t1 = q >> lgcb, c = q & (cb - 1);
        const long long t = ((long long)t1 << lg2) + c0 + c;
        s[pad((c << lg1) + t1)] = wrapped ? load_chirp(chirp, in.n, nf, M, t) : load_in(in, b, chirp, t);
    }
    fft_fwd(s, cb * M1, lg1, tw, lg2);
    double2* Tb = T + b * M;
    for (int q = threadIdx.x; q < cb * M1; q += blockDim.x) {
        const int p = q >> lgcb, c = q & (cb - 1), t2 = c0 + c;
        const unsigned long long m =
            ((unsigned long long)t2 * (unsigned)freq_at(p, lg1)) & (unsigned long long)(M - 1);
        Tb[((long long)p << lg2) + t2] = cmul(s[pad((c << lg1) + p)], twiddle_m(ta, tb, m, lg2));
    }
}

// Launch 2: grid (M1 / rb, traces); rows rb x ... of trace blockIdx.y.
// bhatp == nullptr: forward rows only (the chirp transform's own set-up).
__global__ __launch_bounds__(FFT_TILE_THREADS) void k_fft_rows(double2* __restrict__ T,
                                                               const double2* __restrict__ bhatp, int lg1,
                                                               int lg2, int lgrb, const double2* __restrict__ tw,
                                                               const double2* __restrict__ ta,
                                                               const double2* __restrict__ tb) {
    __shared__ double2 s[padded(1 << FFT_LG_TILE)];
    const int M2 = 1 << lg2, cnt = M2 << lgrb;
    const long long b = blockIdx.y, M = 1ll << (lg1 + lg2);
    const int p0 = blockIdx.x << lgrb;
    double2* row = T + b * M + ((long long)p0 << lg2);
    for (int q = threadIdx.x; q < cnt; q += blockDim.x) s[pad(q)] = row[q];
    fft_fwd(s, cnt, lg2, tw, lg2);
    if (!bhatp) {
        for (int q = threadIdx.x; q < cnt; q += blockDim.x) row[q] = s[pad(q)];
        return;
    }
    const double2* bh = bhatp + ((long long)p0 << lg2);
    for (int q = threadIdx.x; q < cnt; q += blockDim.x) s[pad(q)] = cmul(s[pad(q)], bh[q]);
    fft_inv(s, cnt, lg2, tw, lg2);
    for (int q = threadIdx.x; q < cnt; q += blockDim.x) {
        const int t2 = q & (M2 - 1);
        const unsigned long long m =
            ((unsigned long long)t2 * (unsigned)freq_at(p0 + (q >> lg2), lg1)) & (unsigned long long)(M - 1);
        row[q] = cmulc(s[pad(q)], twiddle_m(ta, tb, m, lg2));
    }
}

// Launch 3: grid (M2 / cb, traces); inverse columns, chirp, first nf out.
__global__ __launch_bounds__(FFT_TILE_THREADS) void k_fft_cols_out(const double2* __restrict__ T,
                                                                   const double2* __restrict__ chirp, int lg1, int lg2,
                                                                   int lgcb, const double2* __restrict__ tw,
                                                                   Spectra out) {
    __shared__ double2 s[padded(1 << FFT_LG_TILE)];
    const int M1 = 1 << lg1, cb = 1 << lgcb;
    const long long b = blockIdx.y, M = 1ll << (lg1 + lg2);
    const int c0 = blockIdx.x << lgcb;
    const double2* Tb = T + b * M;
    for (int q = threadIdx.x; q < cb * M1; q += blockDim.x) {
        const int p = q >> lgcb, c = q & (cb - 1);
        s[pad((c << lg1) + p)] = Tb[((long long)p << lg2) + c0 + c];
    }
    fft_inv(s, cb * M1, lg1, tw, lg2);
    for (int q = threadIdx.x; q < cb * M1; q += blockDim.x) {
        const int t1 = q >> lgcb, c = q & (cb - 1);
        const long long k = ((long long)t1 << lg2) + c0 + c;
        if (k < out.nf) store_out(out, b, k, cmul(s[pad((c << lg1) + t1)], chirp[k]));
    }
}

struct DevBuf {
    void* p = nullptr;
    ~DevBuf() {
        if (p) (void)hipFree(p);
    }
};

int ceil_lg(long long v) {
    int l = 0;
    while ((1ll << l) < v) l++;
    return l;
}

int small_launch(int lg, long long blocks, const Traces& in, const double2* chirp, const double2* bhat,
                 const double2* tw, const Spectra& out, double2* oc) {
    const unsigned threads = (unsigned)std::min(1024, std::max(64, (1 << lg) / 8));
    const dim3 grid((unsigned)blocks);
    if (lg <= 8) hipLaunchKernelGGL(k_fft_small<256>, grid, dim3(threads), 0, nullptr, in, chirp, bhat, lg, tw, out, oc);
    else if (lg <= 11)
        hipLaunchKernelGGL(k_fft_small<2048>, grid, dim3(threads), 0, nullptr, in, chirp, bhat, lg, tw, out, oc);
    else
        hipLaunchKernelGGL(k_fft_small<(1 << FFT_LG_SMALL)>, grid, dim3(threads), 0, nullptr, in, chirp, bhat, lg, tw,
                           out, oc);
    HIPCHK(hipGetLastError());
    return PF_OK;
}

// The transform behind pf_dft and pf_dft_complex: out_im == nullptr stores
// (re, im) pairs to out_re; pairs != 0: in_re holds (re, im) pairs.
int dft_run(const double* in_re, const double* in_im, int pairs, long long batch, long long n, long long nf,
            const double* window, double scale, double* out_re, double* out_im) {
    if (batch < 1 || n < 1 || nf < 1 || nf > n) return fail(PF_ERR_ARG, "need batch, n >= 1 and 1 <= nf <= n");
    if (batch > 65535) return fail(PF_ERR_ARG, "batch must be <= 65535 (got %lld)", batch);
    // n <= 2^(FFT_LG_MAX-1): every length's chirp convolution fits 2^FFT_LG_MAX
    if (n > (1ll << (FFT_LG_MAX - 1)))
        return fail(PF_ERR_ARG, "n = %lld exceeds the longest transform (%lld)", n, (1ll << (FFT_LG_MAX - 1)));
    // a power of two that fits one block: plain FFT of length n; otherwise
    // the chirp form over M >= n + nf - 1 (the four-step path always takes it)
    const int lgn = ceil_lg(n);
    const bool blue = (1ll << lgn) != n || lgn > FFT_LG_SMALL;
    const int lg = blue ? ceil_lg(n + nf - 1) : lgn;
    const long long M = 1ll << lg;
    const bool small = lg <= FFT_LG_SMALL;
    const int lg1 = lg / 2, lg2 = lg - lg1;
    const int tlg = small ? lg : lg2;  // length of the longest FFT pass
    // traces in chunks whose scratch stays within 1 GiB
    const long long chunk = small ? 0 : std::max(1ll, std::min(batch, (1ll << 30) / (M * 16)));

    // one device allocation: tables, input, window, output, scratch
    const int in_step = pairs ? 2 : 1, out_step = out_im ? 1 : 2;
    const size_t in_bytes = (size_t)(batch * n) * in_step * sizeof(double);
    const size_t out_bytes = (size_t)(batch * nf) * out_step * sizeof(double);
    size_t bytes = 0;
    auto room = [&](size_t b) {
        const size_t at = bytes;
        bytes += (b + 255) / 256 * 256;
        return at;
    };
    const size_t o_tw = room(std::max<size_t>(1, ((size_t)1 << tlg) / 2) * sizeof(double2));
    const size_t o_ch = room(blue ? (size_t)n * sizeof(double2) : 0), o_bh = room(blue ? (size_t)M * sizeof(double2) : 0);
    const size_t o_ta = room(small ? 0 : ((size_t)1 << lg1) * sizeof(double2));
    const size_t o_tb = room(small ? 0 : ((size_t)1 << lg2) * sizeof(double2));
    const size_t o_re = room(in_bytes), o_im = room(in_im ? in_bytes : 0);
    const size_t o_win = room(window ? (size_t)n * sizeof(double) : 0);
    const size_t o_ore = room(out_bytes), o_oim = room(out_im ? out_bytes : 0);
    const size_t o_T = room((size_t)(chunk * M) * sizeof(double2));
    DevBuf mem;
    HIPCHK(hipMalloc(&mem.p, bytes));
    char* const base = (char*)mem.p;
    double2* const tw = (double2*)(base + o_tw);
    double2* const ch = blue ? (double2*)(base + o_ch) : nullptr;
    double2* const bh = blue ? (double2*)(base + o_bh) : nullptr;
    double2* const ta = small ? nullptr : (double2*)(base + o_ta);
    double2* const tb = small ? nullptr : (double2*)(base + o_tb);

    const Tables tables = {tw, ch, ta, tb, blue ? n : 0, tlg, lg1, lg2};
    const long long entries = std::max({(1ll << tlg), blue ? n : 0ll, 1ll << lg2});
    hipLaunchKernelGGL(k_fft_tables, dim3((unsigned)((entries + 255) / 256)), dim3(256), 0, nullptr, tables);
    HIPCHK(hipGetLastError());
    int dev = 0, rc;
    HIPCHK(hipGetDevice(&dev));
    if ((rc = copy_in(dev, nullptr, base + o_re, in_re, in_bytes))) return rc;
    if (in_im && (rc = copy_in(dev, nullptr, base + o_im, in_im, in_bytes))) return rc;
    if (window) HIPCHK(hipMemcpy(base + o_win, window, (size_t)n * sizeof(double), hipMemcpyHostToDevice));
    const double* const dre = (const double*)(base + o_re);
    Traces in = {dre, pairs ? dre + 1 : in_im ? (const double*)(base + o_im) : nullptr,
                 window ? (const double*)(base + o_win) : nullptr, n, in_step};
    double* const ore = (double*)(base + o_ore);
    Spectra out = {ore, out_im ? (double*)(base + o_oim) : ore + 1, nf, out_step, blue ? scale / (double)M : scale};

    if (small) {
        if (blue && (rc = small_launch(lg, 1, in, ch, nullptr, tw, out, bh))) return rc;
        if ((rc = small_launch(lg, batch, in, ch, bh, tw, out, nullptr))) return rc;
    } else {
        const int lgcb = FFT_LG_TILE - lg1, lgrb = FFT_LG_TILE - lg2;  // columns / rows per block
        // chirp transform, in the order the rows launch reads
        hipLaunchKernelGGL(k_fft_cols, dim3(1u << (lg2 - lgcb), 1), dim3(FFT_TILE_THREADS), 0, nullptr, in,
                           (const double2*)ch, true, nf, lg1, lg2, lgcb, (const double2*)tw, (const double2*)ta,
                           (const double2*)tb, bh);
        HIPCHK(hipGetLastError());
        hipLaunchKernelGGL(k_fft_rows, dim3(1u << (lg1 - lgrb), 1), dim3(FFT_TILE_THREADS), 0, nullptr, bh,
                           (const double2*)nullptr, lg1, lg2, lgrb, (const double2*)tw, (const double2*)ta,
                           (const double2*)tb);
        HIPCHK(hipGetLastError());
        double2* const T = (double2*)(base + o_T);
        for (long long b0 = 0; b0 < batch; b0 += chunk) {
            const unsigned nb = (unsigned)std::min(chunk, batch - b0);
            Traces ti = in;
            Spectra so = out;
            ti.re += b0 * n * in_step;
            if (ti.im) ti.im += b0 * n * in_step;
            so.re += b0 * nf * out_step;
            so.im += b0 * nf * out_step;
            hipLaunchKernelGGL(k_fft_cols, dim3(1u << (lg2 - lgcb), nb), dim3(FFT_TILE_THREADS), 0, nullptr, ti,
                               (const double2*)ch, false, nf, lg1, lg2, lgcb, (const double2*)tw, (const double2*)ta,
                               (const double2*)tb, T);
            HIPCHK(hipGetLastError());
            hipLaunchKernelGGL(k_fft_rows, dim3(1u << (lg1 - lgrb), nb), dim3(FFT_TILE_THREADS), 0, nullptr, T,
                               (const double2*)bh, lg1, lg2, lgrb, (const double2*)tw, (const double2*)ta,
                               (const double2*)tb);
            HIPCHK(hipGetLastError());
            hipLaunchKernelGGL(k_fft_cols_out, dim3(1u << (lg2 - lgcb), nb), dim3(FFT_TILE_THREADS), 0, nullptr,
                               (const double2*)T, (const double2*)ch, lg1, lg2, lgcb, (const double2*)tw, so);
            HIPCHK(hipGetLastError());
        }
    }
    if ((rc = copy_out(dev, nullptr, out_re, base + o_ore, out_bytes))) return rc;
    if (out_im && (rc = copy_out(dev, nullptr, out_im, base + o_oim, out_bytes))) return rc;
    return PF_OK;
}

}  // namespace

extern "C" int pf_dft(const double* in_re, const double* in_im, int64_t batch, int64_t n, int64_t nf,
                      const double* window, double scale, double* out_re, double* out_im) {
    if (!in_re || !out_re || !out_im) return fail(PF_ERR_ARG, "NULL argument");
    return dft_run(in_re, in_im, 0, batch, n, nf, window, scale, out_re, out_im);
}

extern "C" int pf_dft_complex(const double* in, int32_t in_complex, int64_t batch, int64_t n, int64_t nf,
                              const double* window, double scale, double* out) {
    if (!in || !out) return fail(PF_ERR_ARG, "NULL argument");
    return dft_run(in, nullptr, in_complex ? 1 : 0, batch, n, nf, window, scale, out, nullptr);
}
