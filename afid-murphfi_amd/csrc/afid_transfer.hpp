// afid_transfer.hpp -- transfers between the grids.  Coarse -> refined:
// InterpVelMgrd (InterpVelMgrd.F90:11-237) and InterpTempMultigrid
// (phasefield.F90:498-520); refined -> coarse: k_to_coarse.
//
// Every transfer is a product of one-dimensional 4-point Hermite stencils, so
// the axes can be taken one after the other.
//   k_xfer_x   per coarse column: the coarse gradient (or T) with its wall
//              ghosts, the x stencil, and for vx the sum along x; one row of
//              refined x per coarse column goes to a scratch array.
//   k_xfer_yz  per refined line of one periodic axis, or pair of adjacent
//              ones: walks the other axis, contracts the rows of the 4 (pair:
//              5) coarse lines it reads, keeps the last four in registers for
//              the stencil along the walk, and for vyr / vzr carries the sum
//              along it.
// The x stencil, the only one that crosses lanes, so runs on the coarse columns
// alone (a quarter of the refined ones at ratio 2), and the second kernel is
// whole aligned 16-byte rows of refined x: loads, multiply-adds, stores.
//
// What bounds it: bytes, with the scratch 13 B per refined cell at ratio 2 in
// FP64 (7 in FP32) of which 9 (5) are needed.  Forms that did all three axes
// per tile in LDS or per refined line with lane shuffles were bound by integer
// and lane instructions and by 8-byte loads of mostly clamped lanes; figures of
// both at interp_vel().
#pragma once
#include <hip/hip_runtime.h>
#include "afid_params.hpp"
#include "afid_stencils.hpp"
#include "afid_kernels.hpp"
#include "afid_column.hpp"
#include <type_traits>

namespace afid {

enum XferField { XF_VX = 0, XF_VY = 1, XF_VZ = 2, XF_T = 3 };

// read-only table behind a uniform index: scalar loads
template <typename T>
using ConstTab = const __attribute__((address_space(4))) T *;
template <typename T>
__device__ __forceinline__ ConstTab<T> const_tab(const T *q) { return (ConstTab<T>)(unsigned long long)q; }

template <typename RT, int NR> struct XVec { typedef RT V __attribute__((ext_vector_type(NR))); };

// x part of the transfer of field FLD: D[i][j][kr] (row stride ldxr) for every
// coarse column; for vy / vz also F, the x-transferred velocity of the first
// plane along the field's own axis ([i] for vy, [j] for vz), the start of the
// sums (InterpVelMgrd.F90:93-123, :179-209).  One wavefront per column, walking
// columns with the next one's values already on their way; the coarse values
// of a column (reference x index -1 .. nx+1, wall ghosts InterpVelMgrd.F90:37-51,
// phasefield.F90:502-512) go through LDS to the lanes' refined points (CHR per
// lane), whose weights the workgroup keeps in LDS.
// (CHR * 64 covers the base rows too.)
constexpr int XFX_WAVES = 8;                // at most
template <int CHR, typename RT, int FLD>
__global__ void __launch_bounds__(64 * XFX_WAVES) k_xfer_x(KP p, RT *D, RT *F) {
    using V4 = typename XVec<RT, 4>::V;
    extern __shared__ __align__(16) unsigned char smraw[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const int nxm = p.nxm, nxmr = p.nxmr, len = nxm + 4;
    V4 *wt = reinterpret_cast<V4 *>(smraw);                     // [refined x] the 4 weights
    RT *buf = reinterpret_cast<RT *>(wt + 64 * CHR) + wave * len;       // reference x index xc at buf[xc + 1]
    const RT *xs_w = sel<RT>(p.xs_w, p.xs_wf), *lxa = sel<RT>(p.lxa, p.lxaf);
    for (int k = threadIdx.x; k < 64 * CHR; k += blockDim.x)
        for (int a = 0; a < 4; ++a) reinterpret_cast<RT *>(wt)[4 * k + a] = k < nxmr ? xs_w[4 * k + a] : RT(0);
    RT lx[CHR];
    int xa[CHR];
#pragma unroll
    for (int m = 0; m < CHR; ++m) {
        const int k = lane + 64 * m;
        xa[m] = k < nxmr ? p.xs_src[k] + 1 : 0;
        lx[m] = FLD == XF_VX && k < nxmr ? lxa[k] : RT(0);
    }
    if (lane == 0) { buf[0] = RT(0); buf[len - 1] = RT(0); }
    __syncthreads();
    const double sS = 1 - 2 * p.inslws, sN = 1 - 2 * p.inslwn;
    const long long ncol = (long long)p.ny * p.nz, nw = (long long)gridDim.x * waves;
    const double *f = FLD == XF_VX ? p.vx : FLD == XF_VY ? p.vy : FLD == XF_VZ ? p.vz : p.temp;
    double va[CHR], vb[CHR];                                    // rows k of the column and of its successor (vx: rows k + 1)
    auto fetch = [&](long long col) {
        const int i = int(col / p.ny), j = int(col - (long long)i * p.ny);
        const double *a = f + (long long)i * p.plane + (long long)j * p.ldx;
        const double *b = FLD == XF_VY ? f + (long long)i * p.plane + (long long)wrapp(j, p.ny) * p.ldx
                        : FLD == XF_VZ ? f + (long long)wrapp(i, p.nz) * p.plane + (long long)j * p.ldx : a + 1;
#pragma unroll
        for (int m = 0; m < CHR; ++m) {
            if (64 * m >= nxm) break;
            const int k = min(lane + 64 * m, nxm - 1);
            va[m] = a[k];
            if (FLD != XF_T) vb[m] = b[k];
        }
    };
    auto sync = [] {                                            // LDS of one wavefront
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    long long col = (long long)xcd_block(0) * waves + wave;
    if (col < ncol) fetch(col);
    for (; col < ncol; col += nw) {
        const int i = int(col / p.ny), j = int(col - (long long)i * p.ny);
        const bool first = (FLD == XF_VY && j == 0) || (FLD == XF_VZ && i == 0);
        double tbp = 0.0, ttp = 0.0;
        if (FLD == XF_T) { tbp = p.tempbp[col]; ttp = p.temptp[col]; }
        for (int pass = first ? 1 : 0; pass >= 0; --pass) {
            // pass 0: the gradient (T itself); pass 1: the velocity of the first plane
#pragma unroll
            for (int m = 0; m < CHR; ++m) {
                const int k = lane + 64 * m;
                if (64 * m >= nxm) break;
                double v = va[m];
                if (FLD == XF_VX) v = (vb[m] - v) * p.udx3m[min(k, nxm - 1)];
                else if (FLD != XF_T && !pass) v = (vb[m] - v) * (FLD == XF_VY ? p.dy : p.dz);
                if (k < nxm) {
                    buf[k + 2] = RT(v);
                    if (k == 0) buf[1] = FLD == XF_T ? RT((1.0 - 2.0 * p.tfixs) * v + 2.0 * p.tfixs * tbp) : RT(sS * v);
                    if (k == nxm - 1) buf[nxm + 2] = FLD == XF_T ? RT((1.0 - 2.0 * p.tfixn) * v + 2.0 * p.tfixn * ttp) : RT(sN * v);
                }
            }
            if (!pass && col + nw < ncol) fetch(col + nw);
            sync();
            RT *o = pass ? F + (long long)(FLD == XF_VY ? i : j) * p.ldxr : D + col * p.ldxr;
            RT run = RT(0);
#pragma unroll
            for (int m = 0; m < CHR; ++m) {
                const RT *t = buf + xa[m];
                const V4 w = wt[lane + 64 * m];
                RT v = t[0] * w[0] + t[1] * w[1] + t[2] * w[2] + t[3] * w[3];
                if (FLD == XF_VX) {       // vxr at the face above refined cell k
                    v = run + wave_incl_scan(v * lx[m]);
                    run = wave_lane63(v);
                }
                // (zeros just past the last point: whole vectors of the second kernel)
                const int k = lane + 64 * m;
                if (FLD == XF_VX) { if (k < nxmr) o[k + 1] = v; }
                else if (k < min(nxmr + 3, p.ldxr)) o[k] = v;
            }
            if (FLD == XF_VX && lane == 0) o[0] = RT(0);        // vxr(1) = 0
            sync();
        }
    }
}

// the y / z part of one transfer
struct XferJob {
    const void *D, *F;              // rows of k_xfer_x (F: null for vxr and T)
    void *out;                      // refined field
    const int *s_src, *o_src;       // Hermite sources along the walked (s) and the other (o) axis
    const void *s_w, *o_w;          // weights (RT)
    int nS, nO, cS, cO;             // refined and coarse extents
    long long ds, dq;               // D strides of a coarse step along s and o
    long long rs, ro;               // out strides of a refined step along s and o
    int nx, ld;                     // refined x points, row stride
    int two;                        // the refined steps come two by two: sources s_src[s] = s_src[1] + (s - 1) / 2
    double dl;                      // refined spacing along s
    int nseg;                       // wavefronts that share one walk
};
// value of lane k (uniform) in every lane
__device__ __forceinline__ float lane_value(float v, int k) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), k));
}
__device__ __forceinline__ double lane_value(double v, int k) {
    const long long b = __builtin_bit_cast(long long, v);
    const int lo = __builtin_amdgcn_readlane(int(b), k), hi = __builtin_amdgcn_readlane(int(b >> 32), k);
    return __builtin_bit_cast(double, (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// NL adjacent refined lines per wavefront (their sources span NL + 3 coarse
// lines), NR refined x per lane.  SUM: the walk carries the sum (vyr, vzr).
// With nseg > 1 a workgroup's wavefronts share one walk: each takes a range
// of refined steps; for a sum they first add up their ranges.  The sum runs in
// FP64 also for FP32 fields: an FP32 one rounds the whole value at every step
// (a mean flow of 350 drifts by 2e-4 over 288 steps instead of one rounding of
// 1.5e-5) and left vyr, vzr of a flow without a mean 6% further from FP64.  It
// takes no longer (384 x 384^2 -> 768^3: 3.01 ms a step both).
template <typename RT, int NR, int NL, bool SUM, bool SEG>
__global__ void __launch_bounds__(SEG ? 512 : 256) k_xfer_yz(XferJob jb) {
    using V = typename XVec<RT, NR>::V;
    using VS = typename XVec<std::conditional_t<SUM, double, RT>, NR>::V;     // value of a refined step
    constexpr int NU = NL + 3, PD = 4;                           // coarse lines; coarse steps loaded ahead
    extern __shared__ __align__(32) unsigned char smraw[];
    VS *tot = reinterpret_cast<VS *>(smraw);                     // [seg][line][lane]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nch = (jb.nx + 64 * NR - 1) / (64 * NR), ngr = (jb.nO + NL - 1) / NL;
    // x chunks fastest: neighbouring wavefronts write one row
    const int item = SEG ? int(xcd_block(0)) : int(xcd_block(0)) * 4 + wave;
    const int grp = item / nch, chunk = item - grp * nch, seg = SEG ? wave : 0;
    if (grp >= ngr) return;                      // whole workgroups where they share a walk
    const ConstTab<int> sS = const_tab(jb.s_src), sO = const_tab(jb.o_src);
    const ConstTab<RT> wO = const_tab(static_cast<const RT *>(jb.o_w));
    const int l0 = grp * NL;
    const int o0 = sO[l0] - 1;
    static_assert(!SUM || NL == 1, "a sum walks single lines");
    RT w[NL][4];
    long long ro[NU];
#pragma unroll
    for (int c = 0; c < NU; ++c) ro[c] = (long long)wrapf(o0 + c, jb.cO) * jb.dq;
#pragma unroll
    for (int l = 0; l < NL; ++l) {
        const int ll = min(l0 + l, jb.nO - 1);
#pragma unroll
        for (int c = 0; c < 4; ++c) w[l][c] = wO[4 * ll + c];
    }
    // whether the second line of a pair starts one coarse line after the first:
    // a walk each, so that a line takes its own 4 rows and no fifth with weight
    // 0, which would carry an infinity to where no stencil reads it
    const bool shift = NL == 2 && sO[min(l0 + NL - 1, jb.nO - 1)] - 1 > o0;
    // lanes past the row repeat its last vector (the same values to the same place)
    const int x = min((chunk * 64 + lane) * NR, (jb.nx - 1) / NR * NR);
    const RT *D = static_cast<const RT *>(jb.D);
    // rows of the lines (an odd last line twice, with the same values)
    RT *out[NL];
#pragma unroll
    for (int l = 0; l < NL; ++l) out[l] = static_cast<RT *>(jb.out) + min(l0 + l, jb.nO - 1) * jb.ro + x;
    const double dl = jb.dl;
    auto put = [&](int s, const VS (&v)[NL]) {
#pragma unroll
        for (int l = 0; l < NL; ++l) __builtin_nontemporal_store(__builtin_convertvector(v[l], V), reinterpret_cast<V *>(out[l] + s * jb.rs));
    };
    const int nt = SUM ? jb.nS - 1 : jb.nS;
    const int sa = SEG ? int((long long)nt * seg / jb.nseg) : 0, sb = SEG ? int((long long)nt * (seg + 1) / jb.nseg) : nt;
    VS v[NL];
    // walk of the refined steps sa .. sb - 1
    auto walk = [&](auto store, auto sh) {
        if (sa >= sb) return;
        int cs = sS[sa] - 1;
        const int end = sS[sb - 1] + 2;
        int cw = wrapf(cs, jb.cS);                               // cs on the periodic axis
        V R[PD][NU], W[4][NL];
        auto load = [&](V (&r)[NU]) {
            const RT *q = D + cw * jb.ds;
#pragma unroll
            for (int c = 0; c < NU; ++c) r[c] = *reinterpret_cast<const V *>(q + ro[c] + x);
            if (++cw == jb.cS) cw = 0;
        };
#pragma unroll
        for (int q = 0; q < PD; ++q) load(R[q]);
        // the stencils of 64 refined steps at a time, one per lane
        int s = sa, base = sa, tn = 0;
        RT t0 = RT(0), t1 = RT(0), t2 = RT(0), t3 = RT(0);
        auto fill = [&]() {
            base = s;
            const int k = min(s + lane, sb - 1);
            tn = s + lane < sb ? jb.s_src[k] + 2 : -1 << 30;
            const RT *w4 = static_cast<const RT *>(jb.s_w) + 4 * k;
            t0 = w4[0]; t1 = w4[1]; t2 = w4[2]; t3 = w4[3];
        };
        fill();
        int need = __builtin_amdgcn_readlane(tn, 0);
        auto contract = [&](int q) {
#pragma unroll
            for (int l = 0; l < NL; ++l) {
                // (fixed roundings, those of a chain over all NU rows)
                const int d = l ? int(sh) : 0;
                V P = R[q % PD][1] * w[l][1 - d];
                P = __builtin_elementwise_fma(R[q % PD][2 * d], V(w[l][d]), P);
                P = __builtin_elementwise_fma(R[q % PD][d + 2], V(w[l][2]), P);
                P = __builtin_elementwise_fma(R[q % PD][d + 3], V(w[l][3]), P);
                W[q][l] = P;
            }
        };
        auto emit = [&](int q) {
            const int k = s - base;
            const RT w0 = lane_value(t0, k), w1 = lane_value(t1, k), w2 = lane_value(t2, k), w3 = lane_value(t3, k);
            ++s;
#pragma unroll
            for (int l = 0; l < NL; ++l) {
                const V tv = W[(q + 1) & 3][l] * w0 + W[(q + 2) & 3][l] * w1 + W[(q + 3) & 3][l] * w2 + W[q][l] * w3;
                if constexpr (SUM) v[l] += __builtin_convertvector(tv, VS) * dl;
                else v[l] = tv;
            }
            if (store) put(SUM ? s : s - 1, v);
        };
        for (; cs <= end; cs += 4) {
            if (jb.two && s + 8 <= sb && need == cs && s > 0 && (s & 1)) {
                // ratio 2: every coarse step completes the refined steps s
                // (odd) and s + 1.  Straight-line code, so that a wait for a
                // row counts the stores issued after it instead of draining them.
                if (s - base > 56) fill();
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    contract(q);
                    load(R[q % PD]);
                    emit(q);
                    emit(q);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (s - base > 63) fill();
                need = s < sb ? __builtin_amdgcn_readlane(tn, s - base) : -1 << 30;
                continue;
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (cs + q > end) break;
                contract(q);
                load(R[q % PD]);
                while (need == cs + q) {
                    emit(q);
                    if (s - base > 63 && s < sb) fill();
                    need = s < sb ? __builtin_amdgcn_readlane(tn, s - base) : -1 << 30;
                }
            }
        }
    };
    if (SUM) {
        if (SEG) {
#pragma unroll
            for (int l = 0; l < NL; ++l) v[l] = VS(0);
            walk(std::false_type{}, std::integral_constant<int, 0>{});
#pragma unroll
            for (int l = 0; l < NL; ++l) tot[(seg * NL + l) * 64 + lane] = v[l];
            __syncthreads();
        }
        const RT *F = static_cast<const RT *>(jb.F);
#pragma unroll
        for (int l = 0; l < NL; ++l) v[l] = VS(0);
        if (F)
#pragma unroll
            for (int c = 0; c < NU; ++c) {
                const V f = *reinterpret_cast<const V *>(F + (long long)wrapf(o0 + c, jb.cO) * jb.ld + x);
#pragma unroll
                for (int l = 0; l < NL; ++l) v[l] += __builtin_convertvector(f, VS) * double(w[l][c]);
            }
        if (seg == 0) put(0, v);
        for (int q = 0; SEG && q < seg; ++q)
#pragma unroll
            for (int l = 0; l < NL; ++l) v[l] += tot[(q * NL + l) * 64 + lane];
    }
    if constexpr (NL == 2) {
        if (shift) {
            walk(std::true_type{}, std::integral_constant<int, 1>{});
            return;
        }
    }
    walk(std::true_type{}, std::integral_constant<int, 0>{});
}

// Refined -> coarse cell centres through the fast coarse-grid loop of
// interpolate_xyz_to_coarse_fast (HermiteInterpolations.F90:291-310):
// InterpSalMultigrid (salinity.F90:458-491), InterpPhiMultigrid and the
// transfer of AddLatentHeat (phasefield.F90:470-494, :651-725).
// What is interpolated and where the result goes.
enum CoarseMode {
    CM_SAL = 0,     // S with the wall ghosts of salinity.F90:466-482 -> salc (salc(nx) = 0)
    CM_PHI = 1,     // phi with zero-gradient ghosts (phasefield.F90:479-487) -> phic (phic(nx) = 0)
    CM_LAT = 2      // d phi with zero-gradient ghosts (:674-683) -> out (+)= scale * value
};
// Per axis and coarse index: the first of the 4 refined sources (1-based
// reference index: x may name the wall ghosts 0 and nxr or the zero entries
// beyond them, y/z may name periodic images) and its 4 weights (FP64 for
// k_to_coarse, RT for k_to_coarse_x2).  The
// bracketing (fast) path of interpolate_xyz_to_coarse_fast and the general
// path of interpolate_xyz_to_coarse differ only in these tables.
struct CoarseJob {
    int mode;
    const void *src;            // refined field (RT)
    void *out;                  // coarse field (RT for CM_SAL, double otherwise)
    const int *x_src, *y_src, *z_src;
    const void *x_w, *y_w, *z_w;
    double scale;
    int accumulate;
    int nseg;                   // ranges of coarse z planes
};
// A workgroup takes NL adjacent coarse lines of y and a range of z, its
// wavefronts the refined x (NR per lane).  It walks the refined z planes with
// the rows of the next 2 on their way, contracts the 4 rows of each line
// (NL = 2: lines two refined rows apart share them), keeps the last four
// planes in registers, and where a coarse plane's stencil is complete puts the
// contracted refined row in LDS, from which each thread takes its coarse x.
// Ghosts at the walls are folded into the x weights: the mirrored value into
// the tap it mirrors, the wall's 2 S into gS / gN, whose y / z contraction 16
// lanes form.
// Weights and sums are FP64 also for FP32 fields, so that only what is stored
// is rounded: in FP32 the order y, z, x was up to 5% less accurate (rms) than
// x, y, z at x ratios such as 7/4.  It costs 80 us of 1580 a step at 384 x 384^2
// from 768^3, 1 of 51 at 64 x 96^2 from 128 x 192^2.
// What bounds it: the read of the refined field once (us a launch, at 5.2 TB/s,
// now, and as 64 x 8 x 16 tiles staged in LDS with a barrier per refined plane
// before, which left 72 workgroups at 64^3):
//   64^3 from 128^3 FP64                 4     13     190
//   384 x 192^2 from 768 x 384^2 FP64  196    242     495
//   384 x 384^2 from 768^3 FP32        370    526    1189
//   256^3 from 448 x 512^2 FP32 (phi)  116    145
// Single lines instead of pairs: 1147 against 850 us a step at 384 x 192^2 (8
// rows instead of 6 for two lines), 44 against 50 at 64^3 before the choice of
// ranges (35 now).
template <typename RT, int NR, int NL>
__global__ void __launch_bounds__(512) k_to_coarse(KP p, CoarseJob jb) {
    using V = typename XVec<RT, NR>::V;
    using VD = typename XVec<double, NR>::V;
    constexpr int NU = 4 + 2 * (NL - 1), PD = 2;                // rows; planes loaded ahead (4: the same)
    extern __shared__ __align__(32) unsigned char smraw[];
    double *sm = reinterpret_cast<double *>(smraw);             // [2][line][reference refined x + NR - 1]
    const int LD = (p.nxmr + 3 * NR - 1) / NR * NR;
    const int t = threadIdx.x, T = blockDim.x, lane = t & 63;
    const int ngr = (p.ny + NL - 1) / NL, item = int(xcd_block(0));
    if (item >= ngr * jb.nseg) return;                          // whole workgroups
    const int seg = item / ngr, J0 = (item - seg * ngr) * NL;
    const int I0 = int((long long)p.nz * seg / jb.nseg), I1 = int((long long)p.nz * (seg + 1) / jb.nseg);
    if (I0 >= I1) return;
    const RT *src = static_cast<const RT *>(jb.src);
    const ConstTab<int> sy = const_tab(jb.y_src), sz = const_tab(jb.z_src);
    const ConstTab<double> ywc = const_tab(static_cast<const double *>(jb.y_w));
    const int y0 = sy[J0] - 1, xw = t * NR, x = min(xw, (p.nxmr - 1) / NR * NR);
    double wy[NL][4];
    long long ro[NU];
#pragma unroll
    for (int l = 0; l < NL; ++l)
#pragma unroll
        for (int b = 0; b < 4; ++b) wy[l][b] = ywc[4 * (J0 + l) + b];
#pragma unroll
    for (int c = 0; c < NU; ++c) ro[c] = (long long)wrapf(y0 + c, p.nyr) * p.ldxr + x;
    // taps of coarse k: weights of reference x base .. base + 3, 0 on those
    // outside, where the rows in LDS hold 0 (a clamped base would read points
    // that the stencil does not, and carry an infinity to k)
    struct Taps { int base; double w[4], gS, gN; };
    auto taps = [&](int k) {
        Taps q{1, {0.0, 0.0, 0.0, 0.0}, 0.0, 0.0};
        if (k >= p.nxm) return q;
        const double *w4 = static_cast<const double *>(jb.x_w) + 4 * k;
        const int s = jb.x_src[k];
        q.base = max(-1, min(s, p.nxmr - 1));
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            int kr = s + a;
            double w = w4[a];
            if (kr < 0 || kr > p.nxr) continue;
            if (kr == 0) {
                if (jb.mode == CM_SAL && p.sfixs == 1) { q.gS += w; w = -w; }
            } else if (kr == p.nxr) {
                if (jb.mode == CM_SAL && p.sfixn == 1) { q.gN += w; w = -w; }
            }
            kr = max(1, min(kr, p.nxmr));
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (kr - q.base == c) q.w[c] += w;
        }
        return q;
    };
    Taps tp[2] = {taps(t), taps(t + T)};
    // 2 S of the walls: lane (a, b, l, wall) its point of the y / z stencil
    const bool wall = jb.mode == CM_SAL && (2 * T < p.nxm || __any(tp[0].gS != 0.0 || tp[0].gN != 0.0 || tp[1].gS != 0.0 || tp[1].gN != 0.0));
    const int la = lane & 3, lb = (lane >> 2) & 3, ll = NL == 2 ? (lane >> 4) & 1 : 0;
    const double *bp = lane < 32 ? p.salbp : p.saltp;
    const int by = wrapf(y0 + 2 * ll + lb, p.nyr);
    const double bw = static_cast<const double *>(jb.y_w)[4 * (J0 + ll) + lb];
    double bv = 0.0;
    auto load_wall = [&](int zs) { bv = 2.0 * bp[(long long)wrapf(zs + la, p.nzr) * p.nyr + by]; };

    // (seen by the others after the first barrier of a coarse plane)
    for (int q = t; q < 2 * NL * 4; q += T) {
        const int g = q & 3;                                    // reference x -1, 0, nxmr + 1, nxmr + 2
        sm[(q >> 2) * LD + NR - 1 + (g < 2 ? g - 1 : p.nxmr + g - 1)] = 0.0;
    }

    int zr = sz[I0] - 1;
    const int end = sz[I1 - 1] + 2;
    int zw = wrapf(zr, p.nzr), zl = zr;                          // the plane to load next, on the periodic axis and off it
    V R[PD][NU];
    VD W[4][NL];
    auto load = [&](V (&r)[NU]) {
        const RT *q = src + zw * p.planer;
#pragma unroll
        for (int c = 0; c < NU; ++c) r[c] = *reinterpret_cast<const V *>(q + ro[c]);
        if (zl < end) { ++zl; if (++zw == p.nzr) zw = 0; }       // (past the end: the last plane again)
    };
#pragma unroll
    for (int q = 0; q < PD; ++q) load(R[q]);
    // the stencils of 64 coarse planes at a time, one per lane
    int ic = I0, base = I0, tn = 0;
    double t0 = 0.0, t1 = 0.0, t2 = 0.0, t3 = 0.0;
    auto fill = [&]() {
        base = ic;
        const int k = min(ic + lane, I1 - 1);
        tn = jb.z_src[k] + 2;
        const double *w4 = static_cast<const double *>(jb.z_w) + 4 * k;
        t0 = w4[0]; t1 = w4[1]; t2 = w4[2]; t3 = w4[3];
    };
    fill();
    int need = __builtin_amdgcn_readlane(tn, 0), e = 0;
    if (wall) load_wall(need - 3);
    auto store = [&](long long o, double v) {
        if (jb.mode == CM_SAL) static_cast<RT *>(jb.out)[o] = RT(v);
        else {
            double *out = static_cast<double *>(jb.out);
            const double val = jb.mode == CM_LAT ? jb.scale * v : v;
            out[o] = jb.accumulate ? out[o] + val : val;
        }
    };
    auto emit = [&](int q) {
        const int k = ic - base;
        const double w0 = lane_value(t0, k), w1 = lane_value(t1, k), w2 = lane_value(t2, k), w3 = lane_value(t3, k);
        double *b = sm + (e & 1) * NL * LD;
        e ^= 1;
#pragma unroll
        for (int l = 0; l < NL; ++l) {
            const VD v = W[(q + 1) & 3][l] * w0 + W[(q + 2) & 3][l] * w1 + W[(q + 3) & 3][l] * w2 + W[q][l] * w3;
            double *at = b + l * LD + NR + xw;
            if (xw + NR <= p.nxmr) *reinterpret_cast<VD *>(at) = v;
            else
#pragma unroll
                for (int c = 0; c < NR; ++c)
                    if (xw + c < p.nxmr) at[c] = v[c];
        }
        __syncthreads();
        double g[2][NL] = {};
        if (wall) {
            double s = bv * bw * (la == 0 ? w0 : la == 1 ? w1 : la == 2 ? w2 : w3);
            s += dpp_move<0x128, 0xf, true>(s);                 // row_ror: the 16 points of a line and wall
            s += dpp_move<0x124, 0xf, true>(s);
            s += dpp_move<0x122, 0xf, true>(s);
            s += dpp_move<0x121, 0xf, true>(s);
#pragma unroll
            for (int l = 0; l < NL; ++l) { g[0][l] = lane_value(s, 16 * l); g[1][l] = lane_value(s, 32 + 16 * l); }
        }
        auto point = [&](int kk, const Taps &q) {
            if (kk >= p.nxm) return;
#pragma unroll
            for (int l = 0; l < NL; ++l) {
                const double *r = b + l * LD + NR - 1;
                double v = 0.0;
#pragma unroll
                for (int a = 0; a < 4; ++a) v += r[q.base + a] * q.w[a];
                if (wall) v += q.gS * g[0][l] + q.gN * g[1][l];
                store(bidx(p, kk, J0 + l, ic), v);
            }
        };
        point(t, tp[0]);
        point(t + T, tp[1]);
        for (int kk = t + 2 * T; kk < p.nxm; kk += T) point(kk, taps(kk));
        // salc(nx), phic(nx) stay zero (salinity.F90:463, phasefield.F90:476)
        if (jb.mode != CM_LAT && t < NL) {
            const long long o = bidx(p, p.nxm, J0 + t, ic);
            if (jb.mode == CM_SAL) static_cast<RT *>(jb.out)[o] = RT(0);
            else static_cast<double *>(jb.out)[o] = 0.0;
        }
        ++ic;
    };
    for (; zr <= end; zr += 4) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (zr + q > end) break;
#pragma unroll
            for (int l = 0; l < NL; ++l) {
                const auto row = [&](int b) { return __builtin_convertvector(R[q % PD][2 * l + b], VD); };
                W[q][l] = row(0) * wy[l][0] + row(1) * wy[l][1] + row(2) * wy[l][2] + row(3) * wy[l][3];
            }
            load(R[q % PD]);
            while (need == zr + q) {
                emit(q);
                if (ic >= I1) { need = end + 1; break; }
                if (ic - base > 63) fill();
                need = __builtin_amdgcn_readlane(tn, ic - base);
                if (wall) load_wall(need - 3);
            }
        }
    }
}

// The same for phi and d phi (mirrored ghosts) where every coarse x takes the
// refined 2 k - 1 .. 2 k + 2: the x stencil comes first, on each row as it
// arrives, from a lane's own NR points and one of either neighbour (at the ends
// of a wavefront's run one load more), so that NR / 2 values a lane stay to be
// contracted in y and z and nothing goes through LDS.  As fast as the form
// above (434 / 460 against 429 / 446 us a step, d phi / phi of 512^3 FP32).  It
// is here for its roundings: in FP32 the order x, y, z with dot4 gives phic to
// the bit as the kernel before both did, and the mixed form's melting sphere is
// compared with the FP64 form's after 100 steps, where the kinetic energy of
// the weak flow amplifies round-off (9.6e-7 apart; 1.3e-6 with the exact
// contraction above, which is no worse a solution).  One wavefront per run of
// refined x, pair of lines and range of z.
template <typename RT>
__device__ __forceinline__ RT dot4(RT a0, RT w0, RT a1, RT w1, RT a2, RT w2, RT a3, RT w3) {
    if constexpr (sizeof(RT) == 4) return __builtin_fmaf(a3, w3, __builtin_fmaf(a2, w2, __builtin_fmaf(a0, w0, a1 * w1)));
    else return __builtin_fma(a3, w3, __builtin_fma(a2, w2, __builtin_fma(a0, w0, a1 * w1)));
}
template <typename RT, int NR, int NL>
__global__ void __launch_bounds__(256) k_to_coarse_x2(KP p, CoarseJob jb) {
    using V = typename XVec<RT, NR>::V;
    constexpr int NU = 4 + 2 * (NL - 1), NC = NR / 2, PD = 4;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nch = (p.nxmr + 64 * NR - 1) / (64 * NR), ngr = (p.ny + NL - 1) / NL;
    const int item = int(xcd_block(0)) * 4 + wave;
    if (item >= nch * ngr * jb.nseg) return;
    const int seg = item / (nch * ngr), rest = item - seg * nch * ngr, J0 = rest / nch * NL;
    const int I0 = int((long long)p.nz * seg / jb.nseg), I1 = int((long long)p.nz * (seg + 1) / jb.nseg);
    if (I0 >= I1) return;
    const RT *src = static_cast<const RT *>(jb.src);
    double *out = static_cast<double *>(jb.out);
    const ConstTab<int> sy = const_tab(jb.y_src), sz = const_tab(jb.z_src);
    const ConstTab<RT> ywc = const_tab(static_cast<const RT *>(jb.y_w));
    const int y0 = sy[J0] - 1, xw = ((rest % nch) * 64 + lane) * NR, x = min(xw, (p.nxmr - 1) / NR * NR);
    // the point beyond the run: the mirrored end at the walls
    const int xh = lane == 0 ? max(xw - 1, 0) : lane == 63 ? min(xw + NR, p.nxmr - 1) : x;
    RT wy[NL][4], wx[NC][4];
    long long ro[NU];
#pragma unroll
    for (int l = 0; l < NL; ++l)
#pragma unroll
        for (int b = 0; b < 4; ++b) wy[l][b] = ywc[4 * (J0 + l) + b];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int a = 0; a < 4; ++a) wx[c][a] = static_cast<const RT *>(jb.x_w)[4 * min(xw / 2 + c, p.nxm - 1) + a];
#pragma unroll
    for (int c = 0; c < NU; ++c) ro[c] = (long long)wrapf(y0 + c, p.nyr) * p.ldxr;
    int zr = sz[I0] - 1;
    const int end = sz[I1 - 1] + 2;
    int zw = wrapf(zr, p.nzr), zl = zr;                          // the plane to load next, on the periodic axis and off it
    V R[PD][NU];
    RT H[PD][NU], W[4][NL][NC];
    auto load = [&](V (&r)[NU], RT (&h)[NU]) {
        const RT *q = src + zw * p.planer;
#pragma unroll
        for (int c = 0; c < NU; ++c) { r[c] = *reinterpret_cast<const V *>(q + ro[c] + x); h[c] = q[ro[c] + xh]; }
        if (zl < end) { ++zl; if (++zw == p.nzr) zw = 0; }       // (past the end: the last plane again)
    };
#pragma unroll
    for (int q = 0; q < PD; ++q) load(R[q], H[q]);
    // the stencils of 64 coarse planes at a time, one per lane
    int ic = I0, base = I0, tn = 0;
    RT t0 = RT(0), t1 = RT(0), t2 = RT(0), t3 = RT(0);
    auto fill = [&]() {
        base = ic;
        const int k = min(ic + lane, I1 - 1);
        tn = jb.z_src[k] + 2;
        const RT *w4 = static_cast<const RT *>(jb.z_w) + 4 * k;
        t0 = w4[0]; t1 = w4[1]; t2 = w4[2]; t3 = w4[3];
    };
    fill();
    int need = __builtin_amdgcn_readlane(tn, 0);
    auto contract = [&](int q) {
        RT X[NU][NC];
#pragma unroll
        for (int c = 0; c < NU; ++c) {
            const V v = R[q % PD][c];
            RT a[NR + 2];
            a[0] = pick(lane == 0, H[q % PD][c], lane_prev(RT(v[NR - 1])));
            a[NR + 1] = pick(lane == 63, H[q % PD][c], lane_next(RT(v[0])));
#pragma unroll
            for (int j = 0; j < NR; ++j) a[j + 1] = v[j];
#pragma unroll
            for (int j = 3; j <= NR + 1; j += 2) a[j] = xw + j - 1 == p.nxmr ? a[j - 1] : a[j];      // the mirrored ghost
#pragma unroll
            for (int m = 0; m < NC; ++m) X[c][m] = dot4<RT>(a[2 * m], wx[m][0], a[2 * m + 1], wx[m][1], a[2 * m + 2], wx[m][2], a[2 * m + 3], wx[m][3]);
        }
#pragma unroll
        for (int l = 0; l < NL; ++l)
#pragma unroll
            for (int m = 0; m < NC; ++m)
                W[q][l][m] = dot4<RT>(X[2 * l][m], wy[l][0], X[2 * l + 1][m], wy[l][1], X[2 * l + 2][m], wy[l][2], X[2 * l + 3][m], wy[l][3]);
    };
    auto emit = [&](int q) {
        const int k = ic - base;
        const RT w0 = lane_value(t0, k), w1 = lane_value(t1, k), w2 = lane_value(t2, k), w3 = lane_value(t3, k);
#pragma unroll
        for (int l = 0; l < NL; ++l)
#pragma unroll
            for (int m = 0; m < NC; ++m) {
                const RT v = dot4<RT>(W[(q + 1) & 3][l][m], w0, W[(q + 2) & 3][l][m], w1, W[(q + 3) & 3][l][m], w2, W[q][l][m], w3);
                const int kk = xw / 2 + m;
                const long long o = bidx(p, min(kk, p.nxm), J0 + l, ic);
                const double val = jb.mode == CM_LAT ? jb.scale * double(v) : double(v);
                if (kk < p.nxm) out[o] = jb.accumulate ? out[o] + val : val;
            }
        // phic(nx) stays zero (phasefield.F90:476)
        if (jb.mode != CM_LAT && xw == 0)
#pragma unroll
            for (int l = 0; l < NL; ++l) out[bidx(p, p.nxm, J0 + l, ic)] = 0.0;
        ++ic;
    };
    for (; zr <= end; zr += 4) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (zr + q > end) break;
            contract(q);
            load(R[q % PD], H[q % PD]);
            while (need == zr + q) {
                emit(q);
                if (ic >= I1) { need = end + 1; break; }
                if (ic - base > 63) fill();
                need = __builtin_amdgcn_readlane(tn, ic - base);
            }
        }
    }
}

// index nxr of a refined field to zero
template <typename RT>
__global__ void __launch_bounds__(256) k_zero_tail(RT *f, int n, int ld, long long rows) {
    const long long r = (long long)blockIdx.x * 256 + threadIdx.x;
    if (r < rows) f[r * ld + n] = RT(0);
}

}  // namespace afid
