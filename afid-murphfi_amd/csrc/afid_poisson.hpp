// afid_poisson.hpp -- pressure Poisson solve of SolvePressureCorrection
// (pressure.F90:165-236): real FFT along y, complex FFT along z, one
// wall-normal tridiagonal per Fourier mode, inverse transforms.
//
// Transforms run along the strided y and z directions with the contiguous x
// direction mapped to lanes, so every global access is a run of x-adjacent
// values; a workgroup takes L lines (afid_fft.hpp).  The real y transform
// packs two x-adjacent real lines into one complex line.
//
// Spectral layout: S[i][m][k] (complex, k = x fastest), m = 0..ny/2,
// i = 0..nz-1.  The forward transforms fold in the 1/(ny nz) normalisation
// (pressure.F90:179) and the 1/(al dt) of CalcLocalDivergence.
#pragma once
#include <hip/hip_runtime.h>
#include "afid_params.hpp"
#include "afid_stencils.hpp"
#include "afid_kernels.hpp"
#include "afid_fft.hpp"

namespace afid {

// Transform of an ensemble member's lines, held in LDS from the first stage to
// the last.
//
// LDS layout of L lines of N complex values: element j of line l sits at
// l*S + lpad(j), with one pad element per 32 banks of data (16 FP32 or 8
// FP64 complex values) so the stride-R writes of a Stockham stage spread
// over the banks, and a line stride S = lpad(N)+1 that is not a multiple of
// the 32 banks, so x-adjacent lines (the global-load order) do too.
template <typename R>
__host__ __device__ __forceinline__ int lpad(int i) { return i + (i >> (sizeof(R) == 4 ? 4 : 3)); }
template <typename R>
__host__ __device__ __forceinline__ int line_stride(int n) { return lpad<R>(n) + 1; }

// One Stockham stage of radix RD over L lines of length N held in LDS, by
// the NT threads of the workgroup (L*N <= MAXV*NT).  Each thread keeps
// at most MAXB butterflies of the stage in registers between the read and
// the write phase, so the transform runs in place.
template <int RD, int MAXB, typename R, int NT>
__device__ __forceinline__ void fft_stage(cpx<R> *buf, int L, int N, int S, int Ns, const cpx<R> *tw, int sign) {
    const int nbl = N / RD, nb = L * nbl;
    const FastDiv dnbl(nbl), dns(Ns);
    cpx<R> v[MAXB][RD];
#pragma unroll
    for (int q = 0; q < MAXB; ++q) {
        const int b = threadIdx.x + q * NT;
        if (b < nb) {
            const int line = dnbl.div(b), jj = b - line * nbl;
#pragma unroll
            for (int r = 0; r < RD; ++r) v[q][r] = buf[line * S + lpad<R>(jj + r * nbl)];
        }
    }
    __syncthreads();
    const int tstride = N / (Ns * RD);
#pragma unroll
    for (int q = 0; q < MAXB; ++q) {
        const int b = threadIdx.x + q * NT;
        if (b < nb) {
            const int line = dnbl.div(b), jj = b - line * nbl, jq = dns.div(jj), kk = jj - jq * Ns;
#pragma unroll
            for (int r = 1; r < RD; ++r) {
                cpx<R> w = tw[kk * r * tstride];
                if (sign > 0) w.y = -w.y;
                v[q][r] = cmul(v[q][r], w);
            }
            DftSmall<RD, R>::run(v[q], sign);
            const int dst = jq * Ns * RD + kk;
#pragma unroll
            for (int r = 0; r < RD; ++r) buf[line * S + lpad<R>(dst + r * Ns)] = v[q][r];
        }
    }
    __syncthreads();
}

// Full transform of L lines (L*N <= MAXV*NT), line stride S, radices 8, 4, 2
// and 3, by a workgroup of NT threads.
// MAXV: the most complex values a thread holds in a stage.
template <typename R, int NT, int MAXV>
__device__ __forceinline__ void lds_fft(cpx<R> *buf, int L, int S, const FftPlan<R> &pl, int sign) {
    int Ns = 1;
    for (int s = 0; s < pl.nst; ++s) {
        const int RD = pl.rad[s];
        switch (RD) {
        case 8: fft_stage<8, (MAXV + 7) / 8, R, NT>(buf, L, pl.n, S, Ns, pl.tw, sign); break;
        case 4: fft_stage<4, (MAXV + 3) / 4, R, NT>(buf, L, pl.n, S, Ns, pl.tw, sign); break;
        case 3: fft_stage<3, (MAXV + 2) / 3, R, NT>(buf, L, pl.n, S, Ns, pl.tw, sign); break;
        default: fft_stage<2, (MAXV + 1) / 2, R, NT>(buf, L, pl.n, S, Ns, pl.tw, sign); break;
        }
        Ns *= RD;
    }
}

// Source of the forward transform
enum PoissonSrc { SRC_VELOCITY = 0, SRC_DPH = 1 };

// Divergence (CalcLocalDivergence, pressure.F90:147-161) fused with the real
// forward y transform (pressure.F90:171-174) and the 1/(ny nz) scaling.
// With slot_out, the maximum of |div u| (CheckDivergence units) is also
// reduced into *slot_out; with slots_clear, workgroup 0 zeroes 4 slots.
// Workgroup: 2L x-adjacent real lines (L = 1 << lg complex ones) at one z;
// those of one z, and neighbouring z, whose planes of vz are the same, on one
// XCD.  nbx = ceil(nxm / 2L) workgroups per z.
template <typename R, int MT>
__global__ void __launch_bounds__(MT, fft_waves(MT)) k_div_fft_y(KP p, FftPlan<R> pl, cpx<R> *spec, int lg, int nbx, int src, Gate gate,
                                                        unsigned long long *slot_out, unsigned long long *slots_clear) {
    if (gate_closed(gate)) return;
    extern __shared__ __align__(16) unsigned char smraw[];
    cpx<R> *lb = reinterpret_cast<cpx<R> *>(smraw);
    if (slots_clear && blockIdx.x == 0 && threadIdx.x < 4) slots_clear[threadIdx.x] = 0ull;
    const int item = int(xcd_block(0));
    if (item >= nbx * p.nz) return;
    const int N = p.ny, i = item / nbx, k0 = (item - i * nbx) << (lg + 1);
    const int ip = wrapp(i, p.nz);
    const double usdtal = 1.0 / (p.dt * p.al);
    double dmax = 0.0;
    using P2 = double __attribute__((ext_vector_type(2)));
    const double *vz0 = p.vz + (long long)i * p.plane, *vz1 = p.vz + (long long)ip * p.plane;
    const double *vy0 = p.vy + (long long)i * p.plane, *vx0 = p.vx + (long long)i * p.plane, *dp0 = p.dph + (long long)i * p.plane;
    const auto ld = [&](int line, int j) {
        const int k = k0 + 2 * line;
        if (k >= p.nxm) return mk<R>(R(0), R(0));
        const bool two = k + 1 < p.nxm;
        const int o = j * p.ldx + k;
        if (src == SRC_DPH) return mk<R>(R(dp0[o]), two ? R(dp0[o + 1]) : R(0));
        const P2 z1 = *reinterpret_cast<const P2 *>(vz1 + o), z0 = *reinterpret_cast<const P2 *>(vz0 + o);
        const P2 y1 = *reinterpret_cast<const P2 *>(vy0 + wrapp(j, N) * p.ldx + k), y0 = *reinterpret_cast<const P2 *>(vy0 + o);
        const P2 x0 = *reinterpret_cast<const P2 *>(vx0 + o);
        const double x2 = vx0[o + (two ? 2 : 1)];
        const double da = (z1[0] - z0[0]) * p.dz + (y1[0] - y0[0]) * p.dy + (x0[1] - x0[0]) * p.udx3m[k];
        const double db = two ? (z1[1] - z0[1]) * p.dz + (y1[1] - y0[1]) * p.dy + (x2 - x0[1]) * p.udx3m[k + 1] : 0.0;
        dmax = fmax(dmax, fmax(fabs(da), fabs(db)));
        return mk<R>(R(da * usdtal), R(db * usdtal));
    };
    for (int t = threadIdx.x; t < N << lg; t += blockDim.x) lb[t] = ld(t & ((1 << lg) - 1), t >> lg);
    __syncthreads();
    fft_lines<-1, true, true>(lb, lg, pl, [&](int line, int j) { return lb[(j << lg) + line]; },
                              [&](int line, int j, cpx<R> v) { lb[(j << lg) + line] = v; });
    if (slot_out) {
        dmax = block_max(dmax);
        max_to_slot(slot_out, dmax);
    }
    const R scale = R(1.0 / (double(p.ny) * double(p.nz)));
    for (int t = threadIdx.x; t < p.nymh << lg; t += blockDim.x) {
        const int line = t & ((1 << lg) - 1), m = t >> lg, k = k0 + 2 * line;
        if (k >= p.nxm) continue;
        const cpx<R> zm = lb[(m << lg) + line], zn = lb[((m == 0 ? 0 : N - m) << lg) + line];
        cpx<R> *o = spec + ((long long)i * p.nymh + m) * p.nxm + k;
        // (Z_m + conj Z_{N-m})/2 and (Z_m - conj Z_{N-m})/(2i)
        o[0] = mk<R>(R(0.5) * (zm.x + zn.x) * scale, R(0.5) * (zm.y - zn.y) * scale);
        if (k + 1 < p.nxm) o[1] = mk<R>(R(0.5) * (zm.y + zn.y) * scale, R(-0.5) * (zm.x - zn.x) * scale);
    }
}

// Complex transform along z (pressure.F90:176 forward, :189 backward), in
// place on the spectral array.  Workgroup: L = 1 << lg x-adjacent lines at one
// y-mode m.
template <typename R, int SIGN, int MT>
__global__ void __launch_bounds__(MT, fft_waves(MT)) k_fft_z(KP p, FftPlan<R> pl, cpx<R> *spec, int lg, Gate gate) {
    if (gate_closed(gate)) return;
    extern __shared__ __align__(16) unsigned char smraw[];
    cpx<R> *lb = reinterpret_cast<cpx<R> *>(smraw);
    const int m = blockIdx.y, k0 = blockIdx.x << lg;
    const long long sz = (long long)p.nymh * p.nxm;
    cpx<R> *g = spec + (long long)m * p.nxm + k0;
    const int left = p.nxm - k0;
    fft_lines<SIGN, false, false>(lb, lg, pl,
        [&](int line, int i) { return line < left ? g[i * sz + line] : mk<R>(R(0), R(0)); },
        [&](int line, int i, cpx<R> v) { if (line < left) g[i * sz + line] = v; });
}

// Inverse real y transform (pressure.F90:193-195): two x-adjacent spectra
// A, B (Hermitian, imaginary parts of the m=0 and m=N/2 terms ignored as a
// c2r transform does) become Z = A + iB, whose inverse is a + ib, written
// to dph.
template <typename R, int MT>
__global__ void __launch_bounds__(MT, fft_waves(MT)) k_ifft_y(KP p, FftPlan<R> pl, const cpx<R> *spec, int lg, Gate gate) {
    if (gate_closed(gate)) return;
    extern __shared__ __align__(16) unsigned char smraw[];
    cpx<R> *lb = reinterpret_cast<cpx<R> *>(smraw);
    const int N = p.ny, i = blockIdx.y, k0 = blockIdx.x << (lg + 1);
    for (int t = threadIdx.x; t < p.nymh << lg; t += blockDim.x) {
        const int line = t & ((1 << lg) - 1), m = t >> lg, k = k0 + 2 * line;
        const cpx<R> *row = spec + ((long long)i * p.nymh + m) * p.nxm + k;
        cpx<R> A = k < p.nxm ? row[0] : mk<R>(R(0), R(0));
        cpx<R> B = k + 1 < p.nxm ? row[1] : mk<R>(R(0), R(0));
        if (m == 0 || 2 * m == N) { A.y = R(0); B.y = R(0); }
        lb[(m << lg) + line] = mk<R>(A.x - B.y, A.y + B.x);
        if (m > 0 && N - m > m) lb[((N - m) << lg) + line] = mk<R>(A.x + B.y, B.x - A.y);
    }
    __syncthreads();
    R *out = sel<R>(p.dph, p.dphf) + (long long)i * p.plane + k0;       // dph in the sweep's arithmetic R
    fft_lines<1, true, false>(lb, lg, pl, [&](int line, int j) { return lb[(j << lg) + line]; },
        [&](int line, int j, cpx<R> z) {
            const int k = k0 + 2 * line;
            R *o = out + (long long)j * p.ldx + 2 * line;
            if (k + 1 < p.nxm) *reinterpret_cast<cpx<R> *>(o) = z;
            else if (k < p.nxm) *o = z.x;
        });
}

// Per-mode wall-normal tridiagonal (SolveTridiagonalPressure,
// pressure.F90:201-236) with factors precomputed at set-up.  Modes i and
// nz-i share a matrix (ak1 is even), so one block of two wavefronts solves
// both against one copy of the factors.  grid (nymh, nz/2+1).
template <typename R>
struct PoissonFactors {
    const R *m, *g, *e;   // [mode'][row padded to 64*CH], mode' = m*(nz/2+1) + i'
    int npad;
};
// Solve of one mode's column col (nxm complex values) by one wavefront,
// CH rows per lane, with the factors at fm/fg/fe + fo (rows >= npad read as
// zero, so any CH with 64*CH >= nxm serves).
template <int CH, typename R>
__device__ __forceinline__ void mode_tri_solve(const R *fmp, const R *fgp, const R *fep, long long fo, int npad,
                                               cpx<R> *col, int nxm) {
    const int lane = threadIdx.x & 63;
    R fm[CH], fg[CH], fe[CH];
    cpx<R> v[CH];
#pragma unroll
    for (int q = 0; q < CH; ++q) {
        const int r = lane * CH + q;
        const bool in = r < npad;
        fm[q] = in ? fmp[fo + r] : R(0); fg[q] = in ? fgp[fo + r] : R(0); fe[q] = in ? fep[fo + r] : R(0);
        v[q] = r < nxm ? col[r] : mk<R>(R(0), R(0));
    }
    // forward y_r = d_r - m_r y_{r-1} (complex B, real A)
    R A = R(1);
    cpx<R> Bc = mk<R>(R(0), R(0));
#pragma unroll
    for (int q = 0; q < CH; ++q) { Bc = mk<R>(-fm[q] * Bc.x + v[q].x, -fm[q] * Bc.y + v[q].y); A = -fm[q] * A; }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        R Ap = __shfl_up(A, off, 64), Bx = __shfl_up(Bc.x, off, 64), By = __shfl_up(Bc.y, off, 64);
        if (lane >= off) { Bc = mk<R>(A * Bx + Bc.x, A * By + Bc.y); A = A * Ap; }
    }
    cpx<R> y = mk<R>(__shfl_up(Bc.x, 1, 64), __shfl_up(Bc.y, 1, 64));
    if (lane == 0) y = mk<R>(R(0), R(0));
#pragma unroll
    for (int q = 0; q < CH; ++q) { y = mk<R>(-fm[q] * y.x + v[q].x, -fm[q] * y.y + v[q].y); v[q] = y; }
    // backward x_r = g_r y_r - e_r x_{r+1}
    A = R(1); Bc = mk<R>(R(0), R(0));
#pragma unroll
    for (int q = CH - 1; q >= 0; --q) {
        Bc = mk<R>(-fe[q] * Bc.x + fg[q] * v[q].x, -fe[q] * Bc.y + fg[q] * v[q].y); A = -fe[q] * A;
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        R Ap = __shfl_down(A, off, 64), Bx = __shfl_down(Bc.x, off, 64), By = __shfl_down(Bc.y, off, 64);
        if (lane + off < 64) { Bc = mk<R>(A * Bx + Bc.x, A * By + Bc.y); A = A * Ap; }
    }
    cpx<R> x = mk<R>(__shfl_down(Bc.x, 1, 64), __shfl_down(Bc.y, 1, 64));
    if (lane == 63) x = mk<R>(R(0), R(0));
#pragma unroll
    for (int q = CH - 1; q >= 0; --q) {
        x = mk<R>(-fe[q] * x.x + fg[q] * v[q].x, -fe[q] * x.y + fg[q] * v[q].y); v[q] = x;
    }
#pragma unroll
    for (int q = 0; q < CH; ++q) {
        const int r = lane * CH + q;
        if (r < nxm) col[r] = v[q];
    }
}

template <int CH, typename R>
__global__ void __launch_bounds__(128) k_poisson_tri(KP p, PoissonFactors<R> pf, cpx<R> *spec, Gate gate) {
    if (gate_closed(gate)) return;
    const int wave = threadIdx.x >> 6;
    const int m = blockIdx.x, ih = blockIdx.y, nzh = p.nz / 2 + 1;
    const int i = wave == 0 ? ih : p.nz - ih;
    if (wave == 1 && (ih == 0 || i == ih || i >= p.nz)) return;
    const long long fo = ((long long)m * nzh + ih) * pf.npad;
    mode_tri_solve<CH, R>(pf.m, pf.g, pf.e, fo, pf.npad, spec + ((long long)i * p.nymh + m) * p.nxm, p.nxm);
}

// Set-up of the per-mode factors: one thread per (m, i'), sequential over x.
// Normalised rows (pressure.F90:211-220): a_k = amphk s_k, b = 1+1e-15,
// c_k = apphk s_k, rhs s_k with s_k = 1/(acphk_k - ak2_m - ak1_i).  The
// singular (0,0) mode pins its first unknown to zero instead.
// Stored: m_k = l_k s_{k-1}/s_k, g_k = s_k/u_k, e_k = c_k/u_k so that
// y'_k = d_k - m_k y'_{k-1}, x_k = g_k y'_k - e_k x_{k+1}.
__global__ void k_poisson_factors(KP p, const double *ak1, const double *ak2, double *fm, double *fg, double *fe, int npad) {
    const int nzh = p.nz / 2 + 1;
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long long)p.nymh * nzh) return;
    const int m = int(t / nzh), ih = int(t % nzh);
    const long long fo = t * npad;
    const double K = ak2[m] + ak1[ih];
    const bool gauge = (m == 0 && ih == 0);
    double u_prev = 1.0, c_prev = 0.0, s_prev = 0.0;
    for (int k = 0; k < npad; ++k) {
        if (k >= p.nxm) { fm[fo + k] = 0.0; fg[fo + k] = 0.0; fe[fo + k] = 0.0; continue; }
        double s = 1.0 / (p.acphk[k] - K);
        double a = k > 0 ? p.amphk[k] * s : 0.0;
        double c = k < p.nxm - 1 ? p.apphk[k] * s : 0.0;
        double b = 1.0 + 1.0e-15;
        if (gauge && k == 0) { s = 0.0; a = 0.0; c = 0.0; b = 1.0; }
        double l = k > 0 ? a / u_prev : 0.0;
        double u = b - l * c_prev;
        fm[fo + k] = (k > 0 && s != 0.0) ? l * s_prev / s : 0.0;
        fg[fo + k] = s / u;
        fe[fo + k] = c / u;
        u_prev = u; c_prev = c; s_prev = s;
    }
}

// FP64 -> FP32 copy (factor tables and weights of the mixed form)
__global__ void k_to_float(const double *src, float *dst, long long n) {
    for (long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (long long)gridDim.x * blockDim.x)
        dst[q] = float(src[q]);
}

}  // namespace afid
