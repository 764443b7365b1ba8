// afid_column.hpp -- base column kernel with everything in registers.
//
// Explicit terms of vx, vy, vz, T (+ AddSalBuoyancy, AddCondensation) and
// ImplicitAndUpdateVX/VY/VZ/Temp with their solves (TimeMarcher.F90:45-95).
// LPC lanes of a wavefront own one wall-normal column (64: one column per
// wavefront, 32: two y-adjacent ones); lane l holds the rows 2 LPC g + 2 l
// and + 1 of group g = 0 .. MG-1, so every field access is one aligned 16-byte
// load per lane and the rows above and below a pair come from the
// neighbouring lanes (DPP) or, at a group's ends, from a load of those lanes
// alone.  A group's two rows per lane, the lanes and the groups are in row
// order, so the tridiagonal recurrences run where the rows are: two rows in
// the lane, an affine scan over the lanes, a carry from group to group.  The
// forward sweep follows each group's right-hand sides at once; only its
// results (4 fields x 2 MG values per lane) wait for the backward sweep.
// There is no barrier after the tables are staged.
//
// What bounds it: bytes through the L1 and L2.  k_column_base1 (one row per
// lane, rows changed to a solver layout through LDS) spent its time in the L1:
// an 8-byte load takes as many of its cycles as a 16-byte one, the k-1 / k+1
// rows were loads of their own, and 20 row tables came through it with every
// row.  Here a group's pair takes 29 field loads instead of 130, the tables sit
// in LDS, the old fields wait there for the update instead of being read again
// (32 B per cell that had left the L2), and the arrays touched once (history,
// outputs) are marked so that they do not push the neighbour columns out of the
// L2.  192 x 256^2 in FP64: 897 -> 455 us a launch (1.9 -> 3.8 TB/s of the 136
// B per cell it must move); 256 x 512^2 mixed: 3695 -> 2060 us (104 B per
// cell, 1.9 -> 3.4 TB/s); 384 x 192^2 in FP64: 906 -> 514 us; 64^3: 24 -> 18.6.
#pragma once
#include <hip/hip_runtime.h>
#include "afid_params.hpp"
#include "afid_stencils.hpp"
#include "afid_kernels.hpp"

namespace afid {

// uniform factors of the base terms, rounded as the per-routine kernels round them
template <typename T>
struct BaseConst {
    T dy4, dz4, dy2, dz2;           // dy/4, dz/4, dy/2, dz/2
    T dyqr, dzqr, dyqp, dzqp;       // dy^2, dz^2 over ren / pect
    double alren, alpect, dyal;     // al/ren, al/pect, dy al
};
template <typename T>
static inline BaseConst<T> base_const(const KP &p) {
    BaseConst<T> c;
    c.dy4 = T(p.dy) * T(0.25); c.dz4 = T(p.dz) * T(0.25); c.dy2 = T(p.dy) * T(0.5); c.dz2 = T(p.dz) * T(0.5);
    c.dyqr = T(p.dyq) / T(p.ren); c.dzqr = T(p.dzq) / T(p.ren); c.dyqp = T(p.dyq) / T(p.pect); c.dzqp = T(p.dzq) / T(p.pect);
    c.alren = p.al / p.ren; c.alpect = p.al / p.pect; c.dyal = p.dy * p.al;
    return c;
}

// 16-byte (8-byte for float) pair at a byte offset from a uniform base
template <typename T>
__device__ __forceinline__ typename Pair<T>::T ldp(const T *base, unsigned byte) {
    return *reinterpret_cast<const typename Pair<T>::T *>(reinterpret_cast<const char *>(base) + byte);
}
template <typename T>
__device__ __forceinline__ void stp(T *base, unsigned byte, typename Pair<T>::T v) {
    *reinterpret_cast<typename Pair<T>::T *>(reinterpret_cast<char *>(base) + byte) = v;
}
// the same without keeping the line in L2 (the explicit-term history and the
// outputs are touched once; the L2 is left to the neighbour columns)
template <typename T> struct Native2;
template <> struct Native2<float> { typedef float V __attribute__((ext_vector_type(2))); };
template <> struct Native2<double> { typedef double V __attribute__((ext_vector_type(2))); };
template <typename T>
__device__ __forceinline__ typename Pair<T>::T ldp_nt(const T *base, unsigned byte) {
    using V = typename Native2<T>::V;
    const V v = __builtin_nontemporal_load(reinterpret_cast<const V *>(reinterpret_cast<const char *>(base) + byte));
    typename Pair<T>::T r;
    r.x = v.x; r.y = v.y;
    return r;
}
template <typename T>
__device__ __forceinline__ void stp_nt(T *base, unsigned byte, typename Pair<T>::T v) {
    using V = typename Native2<T>::V;
    V n;
    n.x = v.x; n.y = v.y;
    __builtin_nontemporal_store(n, reinterpret_cast<V *>(reinterpret_cast<char *>(base) + byte));
}
template <typename T>
__device__ __forceinline__ T ld1(const T *base, unsigned byte) {
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + byte);
}

// value of the previous / next lane of the wavefront (wave_shr:1, wave_shl:1)
template <typename T>
__device__ __forceinline__ T lane_prev(T v) { return dpp_move<0x138, 0xf, true>(v); }
template <typename T>
__device__ __forceinline__ T lane_next(T v) { return dpp_move<0x130, 0xf, true>(v); }

// c ? a : b with both sides evaluated by every lane (a lane move inside a
// branch would read lanes that the branch leaves out)
template <typename T>
__device__ __forceinline__ T pick(bool c, T a, T b) { return c ? a : b; }

// v moved by CTRL into the lanes it reaches, old in the others
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_into(double old, double v) {
    const long long b = __builtin_bit_cast(long long, v), o = __builtin_bit_cast(long long, old);
    const int lo = __builtin_amdgcn_update_dpp(int(o), int(b), CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(int(o >> 32), int(b >> 32), CTRL, ROWS, 0xf, false);
    return __builtin_bit_cast(double, (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// Inclusive scans of affine maps y -> A y + B over the LPC lanes of a column,
// NA distinct A's and NB maps (map b uses A ia(b)); the A's of the last step
// are not formed.  Upward: lane order; downward: reverse.
constexpr int kMapA[4] = {0, 1, 1, 2};      // vx, vy, vz, T -> X, YZ, T matrices
template <int CTRL, int ROWS, bool LAST>
__device__ __forceinline__ void scan_step(double (&A)[3], double (&B)[4]) {
#pragma unroll
    for (int f = 0; f < 4; ++f) B[f] = A[kMapA[f]] * dpp_into<CTRL, ROWS>(0.0, B[f]) + B[f];
    if (!LAST)
#pragma unroll
        for (int m = 0; m < 3; ++m) A[m] = A[m] * dpp_into<CTRL, ROWS>(1.0, A[m]);
}
template <int LPC>
__device__ __forceinline__ void scan_up(double (&A)[3], double (&B)[4]) {
    scan_step<0x111, 0xf, false>(A, B);
    scan_step<0x112, 0xf, false>(A, B);
    scan_step<0x114, 0xf, false>(A, B);
    scan_step<0x118, 0xf, false>(A, B);
    scan_step<0x142, 0xa, LPC == 32>(A, B);              // row_bcast:15 into rows 1 and 3
    if (LPC == 64) scan_step<0x143, 0xc, true>(A, B);    // row_bcast:31 into rows 2 and 3
}
template <int LPC>
__device__ __forceinline__ void scan_down(double (&A)[3], double (&B)[4], unsigned lane) {
    scan_step<0x101, 0xf, false>(A, B);
    scan_step<0x102, 0xf, false>(A, B);
    scan_step<0x104, 0xf, false>(A, B);
    scan_step<0x108, 0xf, false>(A, B);
    // rows 0 and 2 take the total of the row above them (its lane 0)
    const int s16 = int((lane & 32) | 16);
    const bool t16 = !(lane & 16);
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        const double b = __shfl(B[f], s16, 64);
        B[f] = A[kMapA[f]] * (t16 ? b : 0.0) + B[f];
    }
    if (LPC == 64) {
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            const double a = __shfl(A[m], s16, 64);
            A[m] = A[m] * (t16 ? a : 1.0);
        }
        const bool t32 = lane < 32;
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            const double b = __shfl(B[f], 32, 64);
            B[f] = A[kMapA[f]] * (t32 ? b : 0.0) + B[f];
        }
    }
}
// value of the column's first / last lane in all its lanes
template <int LPC>
__device__ __forceinline__ double column_last(double v, unsigned lane) {
    if (LPC == 64) return wave_lane63(v);
    return __shfl(v, int(lane | 31), 64);
}
template <int LPC>
__device__ __forceinline__ double column_first(double v, unsigned lane) {
    return __shfl(v, LPC == 64 ? 0 : int(lane & 32), 64);
}

// columns of y per strip, and the workgroups one strip and plane takes
constexpr int COL_STRIP = 16;
template <int LPC, int NW>
constexpr int col_per_block() { return NW * 64 / LPC; }
template <int LPC, int NW>
__host__ __device__ __forceinline__ long long col_blocks(int ny, int nz) {
    return (long long)((ny + COL_STRIP - 1) / COL_STRIP) * (COL_STRIP / col_per_block<LPC, NW>()) * nz;
}
// row tables of the kernel, staged in LDS (LT) or read from global memory
enum ColTab { CT_RK, CT_U3C, CT_U3M, CT_APC, CT_AMC, CT_APS, CT_ACS, CT_AMS, CT_APT, CT_ACT, CT_AMT, CT_LN, CT_SN = CT_LN + 3, CT_E = CT_SN + 3, CT_N = CT_E + 3 };

#define AFID_E(V) (e ? V.y : V.x)
#define AFID_SET(V, VAL) do { if (e) V.y = (VAL); else V.x = (VAL); } while (0)
// keeps the instruction scheduler from moving every load of a group to its
// top: without it the kernel needs 223 to 256 registers and spills
#define AFID_FENCE __builtin_amdgcn_sched_barrier(0);
// WIDE: fields of 4 GiB and more, whose planes take 64-bit bases; the others
// reach a whole field through 32-bit offsets from its start.  With bases for all
// the kernel is 1 to 3% slower (192 x 256^2 FP64 451 -> 459 us a launch, 256 x
// 512^2 mixed 2050 -> 2100): the scalar registers run out.
template <int LPC, int MG, int NW, int KEEP, bool LT, bool WIDE, typename HT>
__global__ void __launch_bounds__(64 * NW) k_column_base_reg(KP p, BaseConst<HT> k, TriFactors fx, TriFactors fyz, TriFactors ft, BaseOut o) {
    using H2 = typename Pair<HT>::T;
    constexpr unsigned ROWS = 2u * LPC * MG;
    __shared__ __align__(16) double tab[LT ? CT_N : 1][LT ? ROWS : 2];
    __shared__ double2 keep[NW][MG][KEEP][64];           // old vx, vy(, vz, T) of the wavefront's columns
    const double *src[CT_N] = {p.rudx3m, p.udx3c, p.udx3m, p.ap3ck, p.am3ck, p.ap3sk, p.ac3sk, p.am3sk, p.ap3ssk, p.ac3ssk, p.am3ssk,
                               fx.ln, fyz.ln, ft.ln, fx.sn, fyz.sn, ft.sn, fx.e, fyz.e, ft.e};
    if (LT) {
#pragma unroll
        for (int q = 0; q < CT_N; ++q)
            for (unsigned r = threadIdx.x; r < ROWS; r += 64u * NW) tab[q][r] = r < unsigned(p.nxm) ? src[q][r] : 0.0;
        __syncthreads();
    }
    const unsigned lane = threadIdx.x & 63, l = lane % LPC;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int CPB = col_per_block<LPC, NW>(), SB = COL_STRIP / CPB;
    const unsigned nxm = p.nxm, rmax = p.ldx - 2;
    const bool use_bref = sizeof(HT) == 4 && p.bref;
    // (without salinity bycs, formed from parameters nobody set, may be infinite or NaN)
    const HT bycs = p.active_s == 1 ? HT(p.bycs) : HT(0);
    const bool lo_lane = l == 0, hi_lane = l == LPC - 1;
    // rows r, r+1 of a table (the global metrics end at row ldx, the factors hold whole groups)
    auto tp = [&](int q, unsigned r) {
        if (LT) return *reinterpret_cast<const double2 *>(&tab[LT ? q : 0][LT ? r : 0]);
        return ldp(src[q], (q < CT_LN ? min(r, rmax) : r) * 8u);
    };
    // each XCD takes a contiguous range of blocks, its workgroups walk it together
    const long long total = col_blocks<LPC, NW>(p.ny, p.nz), perx = (total + 7) / 8;
    const long long b0 = (blockIdx.x % 8) * perx, b1 = min(b0 + perx, total);
#pragma unroll 1
    for (long long blk = b0 + blockIdx.x / 8; blk < b1; blk += gridDim.x / 8) {
    const long long per = (long long)SB * p.nz;
    const int strip = int(blk / per), rem = int(blk - strip * per);
    const int i = rem / SB;
    const int jw = strip * COL_STRIP + (rem % SB) * CPB + wave * (64 / LPC);
    if (jw >= p.ny) continue;
    const bool live = LPC == 64 || jw + int(lane / LPC) < p.ny;
    const int j = live ? jw + int(lane / LPC) : jw;
    const int im = wrapm(i, p.nz), ip = wrapp(i, p.nz);
    // byte offsets into whole FP64 fields (below 4 GiB: the host checks), or
    // into the planes at i - 1, i, i + 1
    const unsigned pl = WIDE ? 0u : unsigned(p.plane) * 8u, row = unsigned(p.ldx) * 8u;
    const unsigned jo = unsigned(j) * row, jmo = unsigned(wrapm(j, p.ny)) * row, jpo = unsigned(wrapp(j, p.ny)) * row;
    const unsigned io = unsigned(i) * pl, imo = unsigned(im) * pl, ipo = unsigned(ip) * pl;
    const unsigned o_c = io + jo, o_jm = io + jmo, o_jp = io + jpo, o_im = imo + jo, o_ip = ipo + jo, o_jpim = imo + jpo, o_jmip = ipo + jmo;
    const long long pc = WIDE ? (long long)i * p.plane : 0, pm = WIDE ? (long long)im * p.plane : 0, pp = WIDE ? (long long)ip * p.plane : 0;
    const double *X = p.vx + pc, *Y = p.vy + pc, *Z = p.vz + pc, *T = p.temp + pc, *P = p.pr + pc;
    const double *Xm = p.vx + pm, *Xp = p.vx + pp, *Ym = p.vy + pm, *Yp = p.vy + pp, *Zm = p.vz + pm, *Zp = p.vz + pp;
    const double *Tm = p.temp + pm, *Tp = p.temp + pp, *Pm = p.pr + pm;
    HT *RX = sel<HT>(p.rux, p.ruxf) + pc, *RY = sel<HT>(p.ruy, p.ruyf) + pc, *RZ = sel<HT>(p.ruz, p.ruzf) + pc, *RT = sel<HT>(p.rut, p.rutf) + pc;
    // (opaque, so that the row tables are read where they are used and not kept in registers from block to block)
    unsigned l2 = 2u * l;
    asm volatile("" : "+v"(l2));
    const double tbp = p.tempbp[(long long)i * p.ny + j], ttp = p.temptp[(long long)i * p.ny + j];

    double y[MG][4][2];
    double cy[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int g = 0; g < MG; ++g) {
        const unsigned r0 = 2u * unsigned(g) * LPC + l2, rb = min(r0, rmax) * 8u, c = o_c + rb;
        // loads of the vx term
        const double2 x = ldp(X, c), v = ldp(Y, c), w = ldp(Z, c), t = ldp(T, c), q = ldp(P, c);
        const double2 xjm = ldp(X, o_jm + rb), xjp = ldp(X, o_jp + rb), xim = ldp(Xm, o_im + rb), xip = ldp(Xp, o_ip + rb);
        const double2 vjp = ldp(Y, o_jp + rb), wip = ldp(Zp, o_ip + rb);
        const unsigned ch = c / 8u * unsigned(sizeof(HT));
        const H2 ox = ldp_nt(RX, ch);
        // the rows just outside the group, by its end lanes
        double ex = 0.0, ev = 0.0, ew = 0.0, et = 0.0, eq = 0.0, exjm = 0.0, exim = 0.0, evjp = 0.0, ewip = 0.0;
        if ((lo_lane && g > 0) || hi_lane) {
            const unsigned eb = hi_lane ? min(r0 + 2u, rmax + 1u) * 8u : rb - 8u;
            ex = ld1(X, o_c + eb); ev = ld1(Y, o_c + eb); ew = ld1(Z, o_c + eb); et = ld1(T, o_c + eb);
            if (hi_lane) { exjm = ld1(X, o_jm + eb); exim = ld1(Xm, o_im + eb); }
            else { eq = ld1(P, o_c + eb); evjp = ld1(Y, o_jp + eb); ewip = ld1(Zp, o_ip + eb); }
        }
        H2 sal;
        sal.x = HT(0); sal.y = HT(0);
        if (p.active_s == 1) sal = ldp(sel<HT>(p.salc, p.salcf) + pc, ch);
        double2 bref = make_double2(0.0, 0.0);
        if (use_bref) bref = ldp(p.bref, rb);
        AFID_FENCE
        // loads of the vy term, in flight over the vx term; vz and T follow alike
        const double2 vjm = ldp(Y, o_jm + rb), vim = ldp(Ym, o_im + rb), vip = ldp(Yp, o_ip + rb);
        const double2 wjm = ldp(Z, o_jm + rb), wjmip = ldp(Zp, o_jmip + rb), qjm = ldp(P, o_jm + rb);
        const H2 oy = ldp_nt(RY, ch);
        AFID_FENCE
        // the two rows' values: V of the pair, of the row below, above
        auto lo2 = [](double b, double2 V) { return make_double2(b, V.x); };
        auto hi2 = [](double2 V, double a) { return make_double2(V.y, a); };
        const bool wx[2] = {r0 >= 1 && r0 < nxm, r0 + 1 < nxm}, wc[2] = {r0 < nxm, r0 + 1 < nxm};
        const bool kl[2] = {r0 == 0, false}, kh[2] = {r0 == nxm - 1, r0 + 1 == nxm - 1};
        double d[4][2];
        {
            // vx: ExplicitTermsVX.F90:42-127, ImplicitAndUpdateVX.F90:37-66
            const double2 rk = tp(CT_RK, r0), u3c = tp(CT_U3C, r0), apc = tp(CT_APC, r0), amc = tp(CT_AMC, r0);
            const double rkb = LT ? tab[CT_RK][LT && r0 ? r0 - 1 : 0] : ld1(p.rudx3m, rb ? rb - 8u : 0u);
            const double2 xk = lo2(pick(lo_lane, ex, lane_prev(x.y)), x), xn = hi2(x, pick(hi_lane, ex, lane_next(x.x)));
            const double2 vk = lo2(pick(lo_lane, ev, lane_prev(v.y)), v), wk = lo2(pick(lo_lane, ew, lane_prev(w.y)), w);
            const double2 tk = lo2(pick(lo_lane, et, lane_prev(t.y)), t), qk = lo2(pick(lo_lane, eq, lane_prev(q.y)), q);
            const HT vjpb = pick(lo_lane, HT(evjp), lane_prev(HT(vjp.y))), wipb = pick(lo_lane, HT(ewip), lane_prev(HT(wip.y)));
            H2 hx;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const HT u3 = HT(AFID_E(u3c)), rkc = HT(AFID_E(rk)), rkm = HT(e ? rk.x : rkb);
                const HT xc = HT(AFID_E(x)), xjm_ = HT(AFID_E(xjm)), xjp_ = HT(AFID_E(xjp)), xim_ = HT(AFID_E(xim)), xip_ = HT(AFID_E(xip));
                const HT vjpk = e ? HT(vjp.x) : vjpb, wipk = e ? HT(wip.x) : wipb;
                const HT hxz = u3 * k.dz4 * ((rkm * wipk + rkc * HT(AFID_E(wip))) * (xip_ + xc) - (rkm * HT(AFID_E(wk)) + rkc * HT(AFID_E(w))) * (xc + xim_));
                const HT hxy = u3 * k.dy4 * ((rkm * vjpk + rkc * HT(AFID_E(vjp))) * (xjp_ + xc) - (rkm * HT(AFID_E(vk)) + rkc * HT(AFID_E(v))) * (xc + xjm_));
                const HT a1 = HT(AFID_E(xn)) + xc, b1 = xc + HT(AFID_E(xk));
                const HT hxx = (a1 * a1 - b1 * b1) * u3 * HT(0.25);
                HT h = -(hxx + hxy + hxz) + (xjm_ - HT(2.0) * xc + xjp_) * k.dyqr + (xim_ - HT(2.0) * xc + xip_) * k.dzqr;
                if (p.gaxis == 1) {
                    // FP32 terms: buoyancy as its deviation from the row's FP64 reference
                    if (use_bref) h += HT(p.byct * (p.active_t * 0.5 * (AFID_E(t) + AFID_E(tk))) - AFID_E(bref));
                    else h += HT(p.byct) * (HT(p.active_t) * HT(0.5) * (HT(AFID_E(t)) + HT(AFID_E(tk))));
                    h -= bycs * AFID_E(sal);
                }
                const double br = AFID_E(bref), px = (AFID_E(q) - AFID_E(qk)) * (p.al * AFID_E(u3c));
                const double dxx = AFID_E(xn) * AFID_E(apc) + AFID_E(x) * (-AFID_E(apc) - AFID_E(amc)) + AFID_E(xk) * AFID_E(amc);
                d[0][e] = wx[e] ? (p.ga * (double(h) + br) + p.ro * (double(AFID_E(ox)) + br) + k.alren * dxx - px) * p.dt : 0.0;
                AFID_SET(hx, wx[e] ? h : AFID_E(ox));     // rows without an equation keep their history
            }
            if (live && r0 < nxm) stp_nt(RX, ch, hx);
        }
        keep[wave][g][0][lane] = x;
        keep[wave][g][1][lane] = v;
        if (KEEP == 4) { keep[wave][g][KEEP - 2][lane] = w; keep[wave][g][KEEP - 1][lane] = t; }
        AFID_FENCE
        const double2 wim = ldp(Zm, o_im + rb), wjp = ldp(Z, o_jp + rb), vjpim = ldp(Ym, o_jpim + rb), qim = ldp(Pm, o_im + rb);
        const H2 oz = ldp_nt(RZ, ch);
        AFID_FENCE
        const double2 u3m = tp(CT_U3M, r0), aps = tp(CT_APS, r0), acs = tp(CT_ACS, r0), ams = tp(CT_AMS, r0);
        {
            // vy: ExplicitTermsVY.F90:50-118, ImplicitAndUpdateVY.F90:41-82
            const double2 vk = lo2(pick(lo_lane, ev, lane_prev(v.y)), v), vn = hi2(v, pick(hi_lane, ev, lane_next(v.x)));
            const double2 xn = hi2(x, pick(hi_lane, ex, lane_next(x.x)));
            const HT xjma = pick(hi_lane, HT(exjm), lane_next(HT(xjm.x)));
            double2 gt = t;
            if (p.gaxis == 2) gt = ldp(T, o_jm + rb);
            H2 hy;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const double dk = kl[e] ? AFID_E(v) : AFID_E(vk), dn = kh[e] ? AFID_E(v) : AFID_E(vn);
                const HT vc = HT(AFID_E(v)), xjmn = e ? xjma : HT(xjm.y), wc_ = HT(AFID_E(w)), wjm_ = HT(AFID_E(wjm));
                const HT vjp_ = HT(AFID_E(vjp)), vjm_ = HT(AFID_E(vjm)), vip_ = HT(AFID_E(vip)), vim_ = HT(AFID_E(vim));
                const HT hyx = ((HT(AFID_E(xn)) + xjmn) * (HT(dn) + vc) - (HT(AFID_E(x)) + HT(AFID_E(xjm))) * (vc + HT(dk))) * HT(AFID_E(u3m)) * HT(0.25);
                const HT a2 = vjp_ + vc, b2 = vjm_ + vc;
                const HT hyy = (a2 * a2 - b2 * b2) * k.dy4;
                const HT hyz = ((vip_ + vc) * (HT(AFID_E(wip)) + HT(AFID_E(wjmip))) - (vc + vim_) * (wc_ + wjm_)) * k.dz4;
                HT h = -(hyx + hyy + hyz) + (vjp_ - HT(2.0) * vc + vjm_) * k.dyqr + (vip_ - HT(2.0) * vc + vim_) * k.dzqr + HT(p.Gy);
                if (p.gaxis == 2) {
                    h += HT(p.byct) * (HT(p.active_t) * HT(0.5) * (HT(AFID_E(t)) + HT(AFID_E(gt))));
                    h -= bycs * AFID_E(sal);
                }
                const double ap = AFID_E(aps), ac = AFID_E(acs), am = AFID_E(ams);
                const double dxv = (kh[e] ? -(ac + am) * p.xplusu * p.inslwn : dn * ap) + AFID_E(v) * ac + (kl[e] ? -(ac + ap) * p.xminusu * p.inslws : dk * am);
                d[1][e] = wc[e] ? (p.ga * double(h) + p.ro * double(AFID_E(oy)) + k.alren * dxv - (AFID_E(q) - AFID_E(qjm)) * k.dyal) * p.dt : 0.0;
                AFID_SET(hy, wc[e] ? h : AFID_E(oy));
            }
            if (live && r0 < nxm) stp_nt(RY, ch, hy);
        }
        AFID_FENCE
        const double2 tjm = ldp(T, o_jm + rb), tjp = ldp(T, o_jp + rb), tim = ldp(Tm, o_im + rb), tip = ldp(Tp, o_ip + rb);
        const H2 ot = ldp_nt(RT, ch);
        AFID_FENCE
        {
            // vz: ExplicitTermsVZ.F90:45-114, ImplicitAndUpdateVZ.F90:38-70
            const double2 wk = lo2(pick(lo_lane, ew, lane_prev(w.y)), w), wn = hi2(w, pick(hi_lane, ew, lane_next(w.x)));
            const double2 xn = hi2(x, pick(hi_lane, ex, lane_next(x.x)));
            const HT xima = pick(hi_lane, HT(exim), lane_next(HT(xim.x)));
            double2 gt = t;
            if (p.gaxis == 3) gt = ldp(Tm, o_im + rb);
            H2 hz;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const double dk = kl[e] ? AFID_E(w) : AFID_E(wk), dn = kh[e] ? AFID_E(w) : AFID_E(wn);
                const HT wc_ = HT(AFID_E(w)), ximn = e ? xima : HT(xim.y), vc = HT(AFID_E(v)), vim_ = HT(AFID_E(vim));
                const HT wip_ = HT(AFID_E(wip)), wim_ = HT(AFID_E(wim)), wjp_ = HT(AFID_E(wjp)), wjm_ = HT(AFID_E(wjm));
                const HT a3 = wip_ + wc_, b3 = wim_ + wc_;
                const HT hzz = (a3 * a3 - b3 * b3) * k.dz4;
                const HT hzy = ((HT(AFID_E(vjp)) + HT(AFID_E(vjpim))) * (wjp_ + wc_) - (vc + vim_) * (wc_ + wjm_)) * k.dy4;
                const HT hzx = ((HT(AFID_E(xn)) + ximn) * (HT(dn) + wc_) - (HT(AFID_E(x)) + HT(AFID_E(xim))) * (wc_ + HT(dk))) * HT(AFID_E(u3m)) * HT(0.25);
                HT h = -(hzx + hzy + hzz) + (wip_ - HT(2.0) * wc_ + wim_) * k.dzqr + (wjp_ - HT(2.0) * wc_ + wjm_) * k.dyqr;
                if (p.gaxis == 3) {
                    h += HT(p.byct) * (HT(p.active_t) * HT(0.5) * (HT(AFID_E(t)) + HT(AFID_E(gt))));
                    h -= bycs * AFID_E(sal);
                }
                const double dxw = dn * AFID_E(aps) + AFID_E(w) * AFID_E(acs) + dk * AFID_E(ams);
                d[2][e] = wc[e] ? (p.ga * double(h) + p.ro * double(AFID_E(oz)) + k.alren * dxw - (AFID_E(q) - AFID_E(qim)) * p.dz * p.al) * p.dt : 0.0;
                AFID_SET(hz, wc[e] ? h : AFID_E(oz));
            }
            if (live && r0 < nxm) stp_nt(RZ, ch, hz);
        }
        AFID_FENCE
        {
            // T: ExplicitTermsTemp.F90:39-77 (wall values above and below the end rows), ImplicitAndUpdateTemp.F90:33-62
            const double2 apt = tp(CT_APT, r0), act = tp(CT_ACT, r0), amt = tp(CT_AMT, r0);
            const double2 tk = lo2(pick(lo_lane, et, lane_prev(t.y)), t), tn = hi2(t, pick(hi_lane, et, lane_next(t.x)));
            const double2 xn = hi2(x, pick(hi_lane, ex, lane_next(x.x)));
            H2 ht;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const HT tc = HT(AFID_E(t));
                const HT tup = kh[e] ? HT(2.0) * HT(ttp) : HT(AFID_E(tn)) + tc, tdn = kl[e] ? HT(2.0) * HT(tbp) : tc + HT(AFID_E(tk));
                const HT tip_ = HT(AFID_E(tip)), tim_ = HT(AFID_E(tim)), tjp_ = HT(AFID_E(tjp)), tjm_ = HT(AFID_E(tjm));
                const HT htx = (HT(AFID_E(xn)) * tup - HT(AFID_E(x)) * tdn) * HT(0.5) * HT(AFID_E(u3m));
                const HT htz = (HT(AFID_E(wip)) * (tip_ + tc) - HT(AFID_E(w)) * (tc + tim_)) * k.dz2;
                const HT hty = (HT(AFID_E(vjp)) * (tjp_ + tc) - HT(AFID_E(v)) * (tc + tjm_)) * k.dy2;
                HT h = -(htx + hty + htz) + (tip_ - HT(2.0) * tc + tim_) * k.dzqp + (tjp_ - HT(2.0) * tc + tjm_) * k.dyqp;
                if (p.moist && wc[e]) h = HT(double(h) + condensation_heat(p, pc + (long long)(o_c / 8u), r0 + e));
                const double ap = AFID_E(apt), ac = AFID_E(act), am = AFID_E(amt);
                const double dxt = (kh[e] ? -(am + ac) * ttp * p.tfixn : AFID_E(tn) * ap) + AFID_E(t) * ac + (kl[e] ? -(ap + ac) * tbp * p.tfixs : AFID_E(tk) * am);
                d[3][e] = wc[e] ? (p.ga * double(h) + p.ro * double(AFID_E(ot)) + k.alpect * dxt) * p.dt : 0.0;
                AFID_SET(ht, wc[e] ? h : AFID_E(ot));
            }
            if (live && r0 < nxm) stp_nt(RT, ch, ht);
        }
        AFID_FENCE
        // forward sweep of the group: y_r = sn_r d_r - ln_r y_{r-1}
        double A[3], ln0[3], ln1[3], B[4];
        double2 sn[3];
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            const double2 ln = tp(CT_LN + m, r0);
            sn[m] = tp(CT_SN + m, r0);
            ln0[m] = ln.x; ln1[m] = ln.y;
            A[m] = ln.x * ln.y;
        }
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            const int m = kMapA[f];
            d[f][0] *= sn[m].x; d[f][1] *= sn[m].y;
            B[f] = d[f][1] - ln1[m] * d[f][0];
            if (g > 0) B[f] = A[m] * (lo_lane ? cy[f] : 0.0) + B[f];
        }
        scan_up<LPC>(A, B);
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            const int m = kMapA[f];
            const double yin = pick(lo_lane, cy[f], lane_prev(B[f]));
            y[g][f][0] = d[f][0] - ln0[m] * yin;
            y[g][f][1] = d[f][1] - ln1[m] * y[g][f][0];
            if (g + 1 < MG) cy[f] = column_last<LPC>(y[g][f][1], lane);
        }
    }
    // backward sweep x_r = y_r - e_r x_{r+1}, top group first, and the update
#pragma unroll
    for (int f = 0; f < 4; ++f) cy[f] = 0.0;
#pragma unroll
    for (int g = MG - 1; g >= 0; --g) {
        const unsigned r0 = 2u * unsigned(g) * LPC + l2, rb = min(r0, rmax) * 8u, c = o_c + rb;
        const double2 u0 = keep[wave][g][0][lane], u1 = keep[wave][g][1][lane];
        const double2 u2 = KEEP == 4 ? keep[wave][g][KEEP - 2][lane] : ldp(Z, c), u3 = KEEP == 4 ? keep[wave][g][KEEP - 1][lane] : ldp(T, c);
        double A[3], B[4];
        double2 e[3];
#pragma unroll
        for (int m = 0; m < 3; ++m) { e[m] = tp(CT_E + m, r0); A[m] = e[m].x * e[m].y; }
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            const int m = kMapA[f];
            B[f] = y[g][f][0] - e[m].x * y[g][f][1];
            if (g + 1 < MG) B[f] = A[m] * (hi_lane ? cy[f] : 0.0) + B[f];
        }
        scan_down<LPC>(A, B, lane);
        double s[4][2];
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            const int m = kMapA[f];
            const double xin = pick(hi_lane, cy[f], lane_next(B[f]));
            s[f][1] = y[g][f][1] - e[m].y * xin;
            s[f][0] = y[g][f][0] - e[m].x * s[f][1];
            if (g > 0) cy[f] = column_first<LPC>(s[f][0], lane);
        }
        if (live && r0 < nxm) {
            const bool in1 = r0 + 1 < nxm;
            // walls of vx: ImplicitAndUpdateVX.F90:86-87; the unused index nx of the others is carried over
            stp_nt(o.vx + pc, c, make_double2(r0 >= 1 ? u0.x + s[0][0] : 0.0, in1 ? u0.y + s[0][1] : 0.0));
            stp_nt(o.vy + pc, c, make_double2(u1.x + s[1][0], in1 ? u1.y + s[1][1] : u1.y));
            stp_nt(o.vz + pc, c, make_double2(u2.x + s[2][0], in1 ? u2.y + s[2][1] : u2.y));
            stp_nt(o.temp + pc, c, make_double2(u3.x + s[3][0], in1 ? u3.y + s[3][1] : u3.y));
        }
    }
    if (live && lo_lane && !(nxm & 1u)) {      // the face nx, alone in its pair when nxm is even
        const unsigned b = o_c + nxm * 8u;
        const double a1 = ld1(Y, b), a2 = ld1(Z, b), a3 = ld1(T, b);
        const long long q = pc + (long long)(b / 8u);
        o.vx[q] = 0.0; o.vy[q] = a1; o.vz[q] = a2; o.temp[q] = a3;
    }
    }
#undef AFID_E
#undef AFID_SET
#undef AFID_FENCE
}

// ---------------------------------------------------------------------------
// refined columns (salinity, phase field) the same way
// ---------------------------------------------------------------------------
// Inclusive scans of one affine map over the LPC lanes of a column.
template <int CTRL, int ROWS, bool LAST>
__device__ __forceinline__ void scan1_step(double &A, double &B) {
    B = A * dpp_into<CTRL, ROWS>(0.0, B) + B;
    if (!LAST) A = A * dpp_into<CTRL, ROWS>(1.0, A);
}
template <int LPC>
__device__ __forceinline__ void scan1_up(double &A, double &B) {
    scan1_step<0x111, 0xf, false>(A, B);
    scan1_step<0x112, 0xf, false>(A, B);
    scan1_step<0x114, 0xf, false>(A, B);
    scan1_step<0x118, 0xf, false>(A, B);
    scan1_step<0x142, 0xa, LPC == 32>(A, B);
    if (LPC == 64) scan1_step<0x143, 0xc, true>(A, B);
}
template <int LPC>
__device__ __forceinline__ void scan1_down(double &A, double &B, unsigned lane) {
    scan1_step<0x101, 0xf, false>(A, B);
    scan1_step<0x102, 0xf, false>(A, B);
    scan1_step<0x104, 0xf, false>(A, B);
    scan1_step<0x108, 0xf, false>(A, B);
    const int s16 = int((lane & 32) | 16);
    const bool t16 = !(lane & 16);
    const double b = __shfl(B, s16, 64);
    B = A * (t16 ? b : 0.0) + B;
    if (LPC == 64) {
        const double a = __shfl(A, s16, 64);
        A = A * (t16 ? a : 1.0);
        const double b2 = __shfl(B, 32, 64);
        B = A * (lane < 32 ? b2 : 0.0) + B;
    }
}
// 16-byte vector access at a byte offset from a uniform base, plain or without keeping the line
template <typename T> struct Native16;
template <> struct Native16<float> { typedef float V __attribute__((ext_vector_type(4))); };
template <> struct Native16<double> { typedef double V __attribute__((ext_vector_type(2))); };
template <typename T>
__device__ __forceinline__ typename Native16<T>::V ld16(const T *base, unsigned byte) {
    return *reinterpret_cast<const typename Native16<T>::V *>(reinterpret_cast<const char *>(base) + byte);
}
template <typename T>
__device__ __forceinline__ typename Native16<T>::V ld16_nt(const T *base, unsigned byte) {
    return __builtin_nontemporal_load(reinterpret_cast<const typename Native16<T>::V *>(reinterpret_cast<const char *>(base) + byte));
}
template <typename T>
__device__ __forceinline__ void st16_nt(T *base, unsigned byte, typename Native16<T>::V v) {
    __builtin_nontemporal_store(v, reinterpret_cast<typename Native16<T>::V *>(reinterpret_cast<char *>(base) + byte));
}

// PHI false: ExplicitSalinity + ImplicitSalinity + SolveImpEqnUpdate_Sal
// (salinity.F90:268-454), the new S to out.  PHI true: ExplicitPhase +
// ImplicitPhase + SolveImpEqnUpdate_Phi (phasefield.F90:345-466), the new phi
// to out and the increment to rhsr (read by AddLatentHeat).  RT: storage and
// explicit-term arithmetic of the refined arrays; the implicit RHS, the solve
// and the update run in FP64.  Layout as k_column_base_reg with NR = 16 /
// sizeof(RT) rows per lane: lane l holds the rows NR (LPC g + l) ...
//
// What bounds it: bytes.  A form that went through LDS to the solver's layout
// waited at two barriers per column and kept 43 to 51 KB of LDS per 4
// wavefronts; the figures of both are at the launch.
template <int LPC, int MG, int NW, typename RT, bool PHI>
__global__ void __launch_bounds__(64 * NW) k_column_refined(KP p, TriFactors f, RT *out) {
    using V = typename Native16<RT>::V;
    constexpr int NR = 16 / sizeof(RT);
    constexpr unsigned ROWS = unsigned(NR) * LPC * MG;
    // row tables: metric (salinity), x operator, folded factors
    enum { T_U3, T_AP, T_AC, T_AM, T_LN, T_SN, T_E, T_N };
    __shared__ __align__(16) double tab[T_N][ROWS];
    {
        const double *src[T_N] = {PHI ? nullptr : p.udx3mr, PHI ? p.ap3spkr : p.ap3sskr, PHI ? p.ac3spkr : p.ac3sskr,
                                  PHI ? p.am3spkr : p.am3sskr, f.ln, f.sn, f.e};
#pragma unroll
        for (int q = PHI ? 1 : 0; q < T_N; ++q)
            for (unsigned r = threadIdx.x; r < ROWS; r += 64u * NW) tab[q][r] = r < unsigned(p.nxmr) ? src[q][r] : 0.0;
    }
    __syncthreads();
    const unsigned lane = threadIdx.x & 63, l = lane % LPC;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int CPB = col_per_block<LPC, NW>(), SB = COL_STRIP / CPB;
    const unsigned n = p.nxmr, rmax = p.ldxr - NR;
    const bool lo_lane = l == 0, hi_lane = l == LPC - 1;
    const RT udy = RT(0.5) * RT(p.dyr), udz = RT(0.5) * RT(p.dzr);
    const RT udyq = PHI ? RT(p.pf_d * p.dyqr) : RT(p.dyqr) / RT(p.pecs), udzq = PHI ? RT(p.pf_d * p.dzqr) : RT(p.dzqr) / RT(p.pecs);
    const double adif = PHI ? p.al * p.pf_d : p.al / p.pecs;
    const long long total = col_blocks<LPC, NW>(p.nyr, p.nzr), perx = (total + 7) / 8;
    const long long b0 = (blockIdx.x % 8) * perx, b1 = min(b0 + perx, total);
#pragma unroll 1
    for (long long blk = b0 + blockIdx.x / 8; blk < b1; blk += gridDim.x / 8) {
        const long long per = (long long)SB * p.nzr;
        const int strip = int(blk / per), rem = int(blk - strip * per);
        const int i = rem / SB, jw = strip * COL_STRIP + (rem % SB) * CPB + wave * (64 / LPC);
        if (jw >= p.nyr) continue;
        const bool live = LPC == 64 || jw + int(lane / LPC) < p.nyr;
        const int j = live ? jw + int(lane / LPC) : jw;
        const long long pc = (long long)i * p.planer, pm = (long long)wrapm(i, p.nzr) * p.planer, pp = (long long)wrapp(i, p.nzr) * p.planer;
        const unsigned row = unsigned(p.ldxr) * unsigned(sizeof(RT));
        const unsigned o_c = unsigned(j) * row, o_jm = unsigned(wrapm(j, p.nyr)) * row, o_jp = unsigned(wrapp(j, p.nyr)) * row;
        const RT *S = (PHI ? sel<RT>(p.phi, p.phif) : sel<RT>(p.sal, p.salf));
        const RT *Sc = S + pc, *Sm = S + pm, *Sp = S + pp;
        const RT *TR = PHI ? sel<RT>(p.tempr, p.temprf) + pc : nullptr;
        const RT *X = PHI ? nullptr : sel<RT>(p.vxr, p.vxrf) + pc, *Y = PHI ? nullptr : sel<RT>(p.vyr, p.vyrf) + pc;
        const RT *Z = PHI ? nullptr : sel<RT>(p.vzr, p.vzrf) + pc, *Zp = PHI ? nullptr : sel<RT>(p.vzr, p.vzrf) + pp;
        RT *RU = (PHI ? sel<RT>(p.ruphi, p.ruphif) : sel<RT>(p.rusal, p.rusalf)) + pc;
        RT *O = out + pc, *D = PHI ? sel<RT>(p.rhsr, p.rhsrf) + pc : nullptr;
        const double sbp = PHI ? 0.0 : p.salbp[(long long)i * p.nyr + j], stp_ = PHI ? 0.0 : p.saltp[(long long)i * p.nyr + j];
        // (opaque: the row tables are read where they are used)
        unsigned lr = unsigned(NR) * l;
        asm volatile("" : "+v"(lr));

        double y[MG][NR];
        V own[MG];
        double cy = 0.0;
#pragma unroll
        for (int g = 0; g < MG; ++g) {
            const unsigned r0 = unsigned(NR) * unsigned(g) * LPC + lr, rb = min(r0, rmax) * unsigned(sizeof(RT)), c = o_c + rb;
            const V s = ld16(Sc, c), sjm = ld16(Sc, o_jm + rb), sjp = ld16(Sc, o_jp + rb), sim = ld16(Sm, c), sip = ld16(Sp, c);
            const V ru = ld16_nt(RU, c);
            V vx{}, vy{}, vyp{}, vz{}, vzp{}, tr{};
            if (PHI) tr = ld16(TR, c);
            else { vx = ld16_nt(X, c); vy = ld16(Y, c); vyp = ld16(Y, o_jp + rb); vz = ld16(Z, c); vzp = ld16(Zp, c); }
            // the rows just outside the group, by its end lanes
            RT es = RT(0), ex = RT(0);
            if ((lo_lane && g > 0) || hi_lane) {
                const unsigned er = hi_lane ? min(r0 + NR, rmax + NR - 1u) : r0 - 1u, eb = o_c + er * unsigned(sizeof(RT));
                es = ld1(Sc, eb);
                if (!PHI && hi_lane) ex = ld1(X, eb);
            }
            own[g] = s;
            const RT sb = pick(lo_lane, es, lane_prev(RT(s[NR - 1]))), sa = pick(hi_lane, es, lane_next(RT(s[0])));
            const RT xa = PHI ? RT(0) : pick(hi_lane, ex, lane_next(RT(vx[0])));
            V h;
            double A = 1.0, B = 0.0;
#pragma unroll
            for (int q = 0; q < NR; ++q) {
                const unsigned k = r0 + q;
                const bool in = k < n, kl = k == 0, kh = k == n - 1;
                const RT sc = s[q], sk = q ? s[q ? q - 1 : 0] : sb, sn = q == NR - 1 ? sa : s[q == NR - 1 ? q : q + 1];
                RT hq;
                if (PHI) {
                    const RT nl = RT(p.pf_b) * sc * (RT(1.0) - sc) * (RT(1.0) - RT(2.0) * sc + RT(p.pf_a) * (tr[q] - RT(p.pf_tm)));
                    hq = (sjp[q] - RT(2.0) * sc + sjm[q]) * udyq + (sip[q] - RT(2.0) * sc + sim[q]) * udzq - nl;
                } else {
                    const RT vc = vx[q], vp = q == NR - 1 ? xa : vx[q == NR - 1 ? q : q + 1];
                    const RT up = kh ? RT(2.0) * RT(stp_) : sn + sc, dn = kl ? RT(2.0) * RT(sbp) : sc + sk;
                    const RT hsx = (vp * up - vc * dn) * RT(tab[T_U3][r0 + q]) * RT(0.5);
                    const RT hsy = (vyp[q] * (sjp[q] + sc) - vy[q] * (sc + sjm[q])) * udy;
                    const RT hsz = (vzp[q] * (sip[q] + sc) - vz[q] * (sc + sim[q])) * udz;
                    hq = -(hsx + hsy + hsz) + (sjp[q] - RT(2.0) * sc + sjm[q]) * udyq + (sip[q] - RT(2.0) * sc + sim[q]) * udzq;
                }
                const double ap = tab[T_AP][r0 + q], ac = tab[T_AC][r0 + q], am = tab[T_AM][r0 + q];
                const double wall = PHI ? 0.0 : 1.0;
                const double dxx = (kh ? -wall * (am + ac) * stp_ * p.sfixn : double(sn) * ap) + double(sc) * ac
                                 + (kl ? -wall * (ap + ac) * sbp * p.sfixs : double(sk) * am);
                const double d = in ? (p.ga * double(hq) + p.ro * double(ru[q]) + adif * dxx) * p.dt : 0.0;
                h[q] = in ? hq : ru[q];                 // rows past the last keep their history
                // forward sweep y_r = sn_r d_r - ln_r y_{r-1}, first with y_{r0-1} = 0
                const double ln = tab[T_LN][r0 + q];
                y[g][q] = d * tab[T_SN][r0 + q];
                B = y[g][q] - ln * B;
                A = -ln * A;
            }
            if (live && r0 < n) st16_nt(RU, c, h);
            if (g > 0) B = A * (lo_lane ? cy : 0.0) + B;
            scan1_up<LPC>(A, B);
            double yr = pick(lo_lane, cy, lane_prev(B));
#pragma unroll
            for (int q = 0; q < NR; ++q) { yr = y[g][q] - tab[T_LN][r0 + q] * yr; y[g][q] = yr; }
            if (g + 1 < MG) cy = column_last<LPC>(yr, lane);
        }
        // backward sweep x_r = y_r - e_r x_{r+1} and the update, top group first
        cy = 0.0;
#pragma unroll
        for (int g = MG - 1; g >= 0; --g) {
            const unsigned r0 = unsigned(NR) * unsigned(g) * LPC + lr, c = o_c + min(r0, rmax) * unsigned(sizeof(RT));
            double A = 1.0, B = 0.0, e[NR];
#pragma unroll
            for (int q = NR - 1; q >= 0; --q) { e[q] = tab[T_E][r0 + q]; B = y[g][q] - e[q] * B; A = -e[q] * A; }
            if (g + 1 < MG) B = A * (hi_lane ? cy : 0.0) + B;
            scan1_down<LPC>(A, B, lane);
            double x = pick(hi_lane, cy, lane_next(B));
            V o, dv;
#pragma unroll
            for (int q = NR - 1; q >= 0; --q) {
                x = y[g][q] - e[q] * x;
                o[q] = r0 + q < n ? RT(double(own[g][q]) + x) : own[g][q];
                dv[q] = RT(x);
            }
            if (g > 0) cy = column_first<LPC>(x, lane);
            if (live && r0 < n) {
                st16_nt(O, c, o);
                if (PHI) {
                    if (r0 + NR <= n) st16_nt(D, c, dv);
                    else
#pragma unroll
                        for (int q = 0; q < NR; ++q)
                            if (r0 + q < n) *reinterpret_cast<RT *>(reinterpret_cast<char *>(D) + c + q * sizeof(RT)) = dv[q];
                }
            }
        }
        if (live && lo_lane && n % NR == 0) {           // the unused index nxr is carried over
            const unsigned b = o_c + n * unsigned(sizeof(RT));
            *reinterpret_cast<RT *>(reinterpret_cast<char *>(O) + b) = ld1(Sc, b);
        }
    }
}

}  // namespace afid
