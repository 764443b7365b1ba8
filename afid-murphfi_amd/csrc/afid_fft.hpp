// afid_fft.hpp -- transforms of x-adjacent strided lines, the butterflies in
// registers.
//
// A workgroup transforms L (a power of two) lines of N = 2^a 3^b complex
// values by Stockham stages of radix 16, 12, 9, 8, 6, 4, 3 or 2.  The first
// stage takes its values from where the caller reads them (global memory), the
// last hands them to where the caller wants them; only between stages they
// pass through LDS.  Lines are fastest over the threads and in LDS (element j
// of line l at j L + l), so that global rows of L values are whole 128-byte
// lines and a row in LDS covers the banks once, whatever the stride of j.
//
// What bounds it: the read and the write of the values, as long as enough of
// them are on their way.  Radices up to 16 make two stages, one pass through
// LDS, of N <= 256, and every thread of the workgroup has a butterfly in every
// stage; with 1024 threads for radix-8 butterflies of 2048 values, values
// copied to LDS before the first stage and from it after the last, three
// quarters of the threads waited at five barriers.  Figures at poisson_sweep().
#pragma once
#include <hip/hip_runtime.h>
#include "afid_params.hpp"

namespace afid {

// complex value of real type R (double in the FP64 form, float in the mixed form)
template <typename R>
struct __align__(2 * sizeof(R)) cpx { R x, y; };
template <typename R>
__device__ __forceinline__ cpx<R> mk(R a, R b) { cpx<R> z; z.x = a; z.y = b; return z; }

constexpr int FFT_STAGES = 14;
template <typename R>
struct FftPlan {
    int n = 1;
    int nst = 0;
    int rad[FFT_STAGES] = {0};
    const cpx<R> *tw = nullptr;   // exp(-2 pi i t/n), t = 0..n-1
};

template <typename R>
__device__ __forceinline__ cpx<R> cmul(cpx<R> a, cpx<R> b) { return mk<R>(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
template <typename R>
__device__ __forceinline__ cpx<R> cadd(cpx<R> a, cpx<R> b) { return mk<R>(a.x + b.x, a.y + b.y); }
template <typename R>
__device__ __forceinline__ cpx<R> csub(cpx<R> a, cpx<R> b) { return mk<R>(a.x - b.x, a.y - b.y); }
// multiply by i*sign
template <typename R>
__device__ __forceinline__ cpx<R> cmulis(cpx<R> a, int sign) { return sign < 0 ? mk<R>(a.y, -a.x) : mk<R>(-a.y, a.x); }

// a exp(sign 2 pi i e / N); e is a constant where this is inlined
template <int N, typename R>
__device__ __forceinline__ cpx<R> cmul_root(cpx<R> a, int e, int sign) {
    constexpr double C16[] = {1.0, 0.92387953251128675613, 0.70710678118654752440, 0.38268343236508977173, 0.0,
                              -0.38268343236508977173, -0.70710678118654752440, -0.92387953251128675613, -1.0, -0.92387953251128675613};
    constexpr double S16[] = {0.0, 0.38268343236508977173, 0.70710678118654752440, 0.92387953251128675613, 1.0,
                              0.92387953251128675613, 0.70710678118654752440, 0.38268343236508977173, 0.0, -0.38268343236508977173};
    constexpr double C12[] = {1.0, 0.86602540378443864676, 0.5, 0.0, -0.5, -0.86602540378443864676, -1.0};
    constexpr double S12[] = {0.0, 0.5, 0.86602540378443864676, 1.0, 0.86602540378443864676, 0.5, 0.0};
    constexpr double C9[] = {1.0, 0.76604444311897803520, 0.17364817766693034885, -0.5, -0.93969262078590838405};
    constexpr double S9[] = {0.0, 0.64278760968653932632, 0.98480775301220805937, 0.86602540378443864676, 0.34202014332566873304};
    if (e == 0) return a;
    if (4 * e == N) return cmulis(a, sign);
    if (2 * e == N) return mk<R>(-a.x, -a.y);
    const double c = N == 16 ? C16[e] : N == 12 ? C12[e] : N == 6 ? C12[2 * e] : C9[e];
    const double s = N == 16 ? S16[e] : N == 12 ? S12[e] : N == 6 ? S12[2 * e] : S9[e];
    return cmul(a, mk<R>(R(c), R(sign < 0 ? -s : s)));
}

template <int N, typename R>
struct DftSmall;
// N = A B: A-point transforms, the roots between, B-point transforms
template <int A, int B, typename R>
__device__ __forceinline__ void dft_split(cpx<R> (&v)[A * B], int sign) {
    cpx<R> t[B][A];
#pragma unroll
    for (int b = 0; b < B; ++b) {
        cpx<R> u[A];
#pragma unroll
        for (int a = 0; a < A; ++a) u[a] = v[B * a + b];
        DftSmall<A, R>::run(u, sign);
#pragma unroll
        for (int a = 0; a < A; ++a) t[b][a] = cmul_root<A * B>(u[a], a * b, sign);
    }
#pragma unroll
    for (int a = 0; a < A; ++a) {
        cpx<R> u[B];
#pragma unroll
        for (int b = 0; b < B; ++b) u[b] = t[b][a];
        DftSmall<B, R>::run(u, sign);
#pragma unroll
        for (int b = 0; b < B; ++b) v[a + A * b] = u[b];
    }
}
template <typename R>
struct DftSmall<1, R> {
    static __device__ __forceinline__ void run(cpx<R> (&)[1], int) {}
};
template <typename R>
struct DftSmall<2, R> {
    static __device__ __forceinline__ void run(cpx<R> (&v)[2], int) {
        cpx<R> a = v[0], b = v[1];
        v[0] = cadd(a, b); v[1] = csub(a, b);
    }
};
template <typename R>
struct DftSmall<3, R> {
    static __device__ __forceinline__ void run(cpx<R> (&v)[3], int sign) {
        const R s3 = R(0.86602540378443864676);   // sin(2 pi/3)
        cpx<R> t1 = cadd(v[1], v[2]), t2 = csub(v[1], v[2]);
        cpx<R> m = mk<R>(v[0].x - R(0.5) * t1.x, v[0].y - R(0.5) * t1.y);
        cpx<R> r = cmulis(mk<R>(s3 * t2.x, s3 * t2.y), sign);
        v[0] = cadd(v[0], t1);
        v[1] = cadd(m, r);
        v[2] = csub(m, r);
    }
};
template <typename R>
struct DftSmall<4, R> {
    static __device__ __forceinline__ void run(cpx<R> (&v)[4], int sign) {
        cpx<R> a = cadd(v[0], v[2]), b = csub(v[0], v[2]), c = cadd(v[1], v[3]), d = cmulis(csub(v[1], v[3]), sign);
        v[0] = cadd(a, c); v[2] = csub(a, c);
        v[1] = cadd(b, d); v[3] = csub(b, d);
    }
};
template <typename R>
struct DftSmall<8, R> {
    static __device__ __forceinline__ void run(cpx<R> (&v)[8], int sign) {
        const R h = R(0.70710678118654752440);    // 1/sqrt(2)
        cpx<R> e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
        DftSmall<4, R>::run(e, sign);
        DftSmall<4, R>::run(o, sign);
        // w8^k = exp(sign 2 pi i k/8)
        cpx<R> w1 = mk<R>(h, R(sign) * h), w3 = mk<R>(-h, R(sign) * h);
        cpx<R> t0 = o[0], t1 = cmul(o[1], w1), t2 = cmulis(o[2], sign), t3 = cmul(o[3], w3);
        v[0] = cadd(e[0], t0); v[4] = csub(e[0], t0);
        v[1] = cadd(e[1], t1); v[5] = csub(e[1], t1);
        v[2] = cadd(e[2], t2); v[6] = csub(e[2], t2);
        v[3] = cadd(e[3], t3); v[7] = csub(e[3], t3);
    }
};
template <typename R>
struct DftSmall<6, R> { static __device__ __forceinline__ void run(cpx<R> (&v)[6], int sign) { dft_split<2, 3>(v, sign); } };
template <typename R>
struct DftSmall<9, R> { static __device__ __forceinline__ void run(cpx<R> (&v)[9], int sign) { dft_split<3, 3>(v, sign); } };
template <typename R>
struct DftSmall<12, R> { static __device__ __forceinline__ void run(cpx<R> (&v)[12], int sign) { dft_split<4, 3>(v, sign); } };
template <typename R>
struct DftSmall<16, R> { static __device__ __forceinline__ void run(cpx<R> (&v)[16], int sign) { dft_split<4, 4>(v, sign); } };

// Division by a workgroup-uniform d through one multiply: whenever x * d <=
// 2^32, floor(x / d) = umulhi(x, ceil(2^32 / d)) (the error term, below
// x / 2^32 <= 1/d, never reaches the next integer, since frac(x/d) <= 1 - 1/d).
// d = 1 is passed through.
struct FastDiv {
    unsigned d, m;
    __device__ __forceinline__ explicit FastDiv(unsigned d_) : d(d_), m(d_ > 1 ? 0xFFFFFFFFu / d_ + 1u : 0u) {}
    __device__ __forceinline__ unsigned div(unsigned x) const { return d == 1 ? x : __umulhi(x, m); }
};

// Threads of a workgroup, at most, and the registers that go with them: the
// butterflies in FP64 take 160, three wavefronts per SIMD, where a workgroup
// has up to 512 threads; larger ones have 128 and keep some values in scratch
// (z transform of 192 x 256^2: 51 us a launch in scratch, 45 in registers).
constexpr int FFT_MAXT = 1024;
constexpr int fft_waves(int mt) { return mt > 512 ? 4 : 3; }
// Threads for L lines: one butterfly a thread in the stages of the smallest
// radix above 8 (else of the largest radix).  A stage of radix 8 has then at
// most 2 a thread, one of a smaller RD at most ceil(12 / RD).
inline int fft_threads(int n, int nst, const int *rad, int L) {
    int least = 0, most = 1;
    bool small = false;
    for (int s = 0; s < nst; ++s) {
        most = most > rad[s] ? most : rad[s];
        if (rad[s] > 8 && (!least || rad[s] < least)) least = rad[s];
        if (rad[s] < 8) small = true;
    }
    const int per = !least ? most : small && least > 12 ? 12 : least;
    return ((L * n + per - 1) / per + 63) / 64 * 64;
}

// One stage: butterflies of the values ld(line, j), results to st(line, j, v).
template <int RD, int SIGN, bool FIRST, bool FROM, bool TO, typename R, typename LD, typename ST>
__device__ __forceinline__ void fft_stage_reg(int lg, int N, int Ns, const cpx<R> *tw, LD ld, ST st) {
    constexpr int MAXB = RD > 8 || RD == 1 ? 1 : RD == 8 ? 2 : (12 + RD - 1) / RD;
    const int nbl = N / RD, nb = nbl << lg, T = blockDim.x, t = threadIdx.x, lm = (1 << lg) - 1;
    cpx<R> v[MAXB][RD];
#pragma unroll
    for (int q = 0; q < MAXB; ++q) {
        const int b = t + q * T;
        if (b < nb) {
#pragma unroll
            for (int r = 0; r < RD; ++r) v[q][r] = ld(b & lm, (b >> lg) + r * nbl);
        }
    }
    if (FROM && TO) __syncthreads();                 // LDS is read before it is written again
    const FastDiv dns(Ns);
    const int tstride = N / (Ns * RD);
#pragma unroll
    for (int q = 0; q < MAXB; ++q) {
        const int b = t + q * T;
        if (b < nb) {
            const int jj = b >> lg, jq = dns.div(jj), kk = jj - jq * Ns;
            if (!FIRST) {                            // (the first stage has no roots)
#pragma unroll
                for (int r = 1; r < RD; ++r) {
                    cpx<R> w = tw[kk * r * tstride];
                    if (SIGN > 0) w.y = -w.y;
                    v[q][r] = cmul(v[q][r], w);
                }
            }
            DftSmall<RD, R>::run(v[q], SIGN);
            const int dst = jq * Ns * RD + kk;
#pragma unroll
            for (int r = 0; r < RD; ++r) st(b & lm, dst + r * Ns, v[q][r]);
        }
    }
    if (TO) __syncthreads();
}
template <int SIGN, bool FIRST, bool FROM, bool TO, typename R, typename LD, typename ST>
__device__ __forceinline__ void fft_stage_any(int RD, int lg, int N, int Ns, const cpx<R> *tw, LD ld, ST st) {
    switch (RD) {
    case 16: fft_stage_reg<16, SIGN, FIRST, FROM, TO>(lg, N, Ns, tw, ld, st); break;
    case 12: fft_stage_reg<12, SIGN, FIRST, FROM, TO>(lg, N, Ns, tw, ld, st); break;
    case 9: fft_stage_reg<9, SIGN, FIRST, FROM, TO>(lg, N, Ns, tw, ld, st); break;
    case 8: fft_stage_reg<8, SIGN, FIRST, FROM, TO>(lg, N, Ns, tw, ld, st); break;
    case 6: fft_stage_reg<6, SIGN, FIRST, FROM, TO>(lg, N, Ns, tw, ld, st); break;
    case 4: fft_stage_reg<4, SIGN, FIRST, FROM, TO>(lg, N, Ns, tw, ld, st); break;
    case 3: fft_stage_reg<3, SIGN, FIRST, FROM, TO>(lg, N, Ns, tw, ld, st); break;
    case 2: fft_stage_reg<2, SIGN, FIRST, FROM, TO>(lg, N, Ns, tw, ld, st); break;
    default: fft_stage_reg<1, SIGN, FIRST, FROM, TO>(lg, N, Ns, tw, ld, st); break;
    }
}
// Transform of 1 << lg lines: values from ld(line, j) to st(line, j, v), buf
// between (N << lg values).  SRC / DST: ld reads / st writes buf itself (filled
// before a barrier; the last store is followed by one).
template <int SIGN, bool SRC, bool DST, typename R, typename LD, typename ST>
__device__ __forceinline__ void fft_lines(cpx<R> *buf, int lg, const FftPlan<R> &pl, LD ld, ST st) {
    const auto get = [&](int line, int j) { return buf[(j << lg) + line]; };
    const auto put = [&](int line, int j, cpx<R> v) { buf[(j << lg) + line] = v; };
    if (pl.nst <= 1) {
        fft_stage_any<SIGN, true, SRC, DST>(pl.nst ? pl.rad[0] : 1, lg, pl.n, 1, pl.tw, ld, st);
        return;
    }
    fft_stage_any<SIGN, true, SRC, true>(pl.rad[0], lg, pl.n, 1, pl.tw, ld, put);
    int Ns = pl.rad[0];
    for (int s = 1; s + 1 < pl.nst; ++s) {
        fft_stage_any<SIGN, false, true, true>(pl.rad[s], lg, pl.n, Ns, pl.tw, get, put);
        Ns *= pl.rad[s];
    }
    fft_stage_any<SIGN, false, true, DST>(pl.rad[pl.nst - 1], lg, pl.n, Ns, pl.tw, get, st);
}

}  // namespace afid
