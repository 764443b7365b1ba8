// afid_kernels.hpp -- HIP kernels of the substep (except the Poisson
// transforms, in afid_poisson.hpp).
//
// Point kernels: block (64,4), thread (k, j) with x fastest so a wavefront
// reads 64 consecutive doubles; grid (ceil(n/64), ceil(ny/4), nz).
// Column kernels: one 64-lane wavefront per wall-normal column, each lane
// owning CH consecutive rows; the tridiagonal recurrences run as two
// wavefront-wide affine scans (forward elimination, back substitution).
#pragma once
#include <hip/hip_runtime.h>
#include "afid_params.hpp"
#include "afid_stencils.hpp"

namespace afid {

#define AFID_POINT_PROLOGUE(NXLIM, NY, NZ)                                    \
    const int k = blockIdx.x * 64 + threadIdx.x;                               \
    const int j = blockIdx.y * 4 + threadIdx.y;                                \
    const int i = blockIdx.z;                                                  \
    if (k >= (NXLIM) || j >= (NY)) return;                                     \
    const int jm = wrapm(j, NY), jp = wrapp(j, NY), im = wrapm(i, NZ), ip = wrapp(i, NZ); \
    (void)jm; (void)jp; (void)im; (void)ip;

// Refinement gate of the mixed form: a launch of a refinement sweep whose
// gate slot holds a divergence at or below tol returns at once.  Slots hold
// the bit pattern of a non-negative double (ordered like the value).
struct Gate {
    const unsigned long long *slot;   // null: always run
    double tol;
};
__device__ __forceinline__ bool gate_closed(const Gate &g) {
    return g.slot && __longlong_as_double((long long)*g.slot) <= g.tol;
}

// block-wide reductions (result valid in thread 0)
__device__ __forceinline__ double block_max(double v) {
    __shared__ double sm[16];
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_down(v, off, 64));
    const int t = threadIdx.x + threadIdx.y * blockDim.x, w = t >> 6;
    if ((t & 63) == 0) sm[w] = v;
    __syncthreads();
    const int nw = (blockDim.x * blockDim.y + 63) >> 6;
    if (t == 0) { double m = sm[0]; for (int q = 1; q < nw; ++q) m = fmax(m, sm[q]); v = m; }
    return v;
}
__device__ __forceinline__ double block_sum(double v) {
    __shared__ double ss[16];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    const int t = threadIdx.x + threadIdx.y * blockDim.x, w = t >> 6;
    if ((t & 63) == 0) ss[w] = v;
    __syncthreads();
    const int nw = (blockDim.x * blockDim.y + 63) >> 6;
    if (t == 0) { double m = ss[0]; for (int q = 1; q < nw; ++q) m += ss[q]; v = m; }
    __syncthreads();
    return v;
}

// thread 0 of a workgroup folds its maximum into a slot; the atomic is
// skipped when the slot already holds at least that value (the plain read
// may be stale, which only costs an atomic), so a grid of many workgroups
// does not serialise on one address
__device__ __forceinline__ void max_to_slot(unsigned long long *slot, double v) {
    if (threadIdx.x == 0 && threadIdx.y == 0) {
        const unsigned long long bits = (unsigned long long)__double_as_longlong(v);
        if (bits > *slot) atomicMax(slot, bits);
    }
}

// ---------------------------------------------------------------------------
// per-routine explicit kernels
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_explicit_vx(KP p) {
    AFID_POINT_PROLOGUE(p.nxm, p.ny, p.nz)
    if (k == 0) return;   // qcap(1) is not computed (ExplicitTermsVX.F90:50)
    const Nb n = make_nb(p, j, i);
    p.qcap[bidx(p, k, j, i)] = ex_vx<double>(p, n, k);
}
__global__ void __launch_bounds__(256) k_explicit_vy(KP p) {
    AFID_POINT_PROLOGUE(p.nxm, p.ny, p.nz)
    const Nb n = make_nb(p, j, i);
    p.dph[bidx(p, k, j, i)] = ex_vy<double>(p, n, k);
}
__global__ void __launch_bounds__(256) k_explicit_vz(KP p) {
    AFID_POINT_PROLOGUE(p.nxm, p.ny, p.nz)
    const Nb n = make_nb(p, j, i);
    p.dq[bidx(p, k, j, i)] = ex_vz<double>(p, n, k);
}
__global__ void __launch_bounds__(256) k_explicit_temp(KP p) {
    AFID_POINT_PROLOGUE(p.nxm, p.ny, p.nz)
    const Nb n = make_nb(p, j, i);
    p.hro[bidx(p, k, j, i)] = ex_temp<double>(p, n, k);
}
__global__ void __launch_bounds__(256) k_explicit_sal(KP p) {
    AFID_POINT_PROLOGUE(p.nxmr, p.nyr, p.nzr)
    const NbS<double> n = make_nbs<double>(p, j, i);
    p.hsal[ridx(p, k, j, i)] = ex_sal<double, double>(p, n, k);
}
// AddSalBuoyancy, salinity.F90:495-506
__global__ void __launch_bounds__(256) k_add_sal_buoyancy(KP p, double *rkv) {
    AFID_POINT_PROLOGUE(p.nxm, p.ny, p.nz)
    const long long c = bidx(p, k, j, i);
    rkv[c] = rkv[c] - p.bycs * p.salc[c];
}

// ---------------------------------------------------------------------------
// per-routine implicit RHS kernels (ImplicitAndUpdate*.F90 loops)
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_rhs_vx(KP p) {
    AFID_POINT_PROLOGUE(p.nxm, p.ny, p.nz)
    if (k == 0) return;
    const long long c = bidx(p, k, j, i);
    const double h = p.qcap[c];
    const Nb n = make_nb(p, j, i);
    p.rhsx[c] = rhs_vx(p, n, h, p.rux[c], k);
    p.rux[c] = h;
}
__global__ void __launch_bounds__(256) k_rhs_vy(KP p) {
    AFID_POINT_PROLOGUE(p.nxm, p.ny, p.nz)
    const long long c = bidx(p, k, j, i);
    const double h = p.dph[c];
    const Nb n = make_nb(p, j, i);
    p.rhsy[c] = rhs_vy(p, n, h, p.ruy[c], k);
    p.ruy[c] = h;
}
__global__ void __launch_bounds__(256) k_rhs_vz(KP p) {
    AFID_POINT_PROLOGUE(p.nxm, p.ny, p.nz)
    const long long c = bidx(p, k, j, i);
    const double h = p.dq[c];
    const Nb n = make_nb(p, j, i);
    p.rhsz[c] = rhs_vz(p, n, h, p.ruz[c], k);
    p.ruz[c] = h;
}
__global__ void __launch_bounds__(256) k_rhs_temp(KP p) {
    AFID_POINT_PROLOGUE(p.nxm, p.ny, p.nz)
    const long long c = bidx(p, k, j, i);
    const double h = p.hro[c];
    const Nb n = make_nb(p, j, i);
    p.rhst[c] = rhs_temp(p, n, h, p.rut[c], k);
    p.rut[c] = h;
}
__global__ void __launch_bounds__(256) k_rhs_sal(KP p) {
    AFID_POINT_PROLOGUE(p.nxmr, p.nyr, p.nzr)
    const long long c = ridx(p, k, j, i);
    const double h = p.hsal[c];
    const NbS<double> n = make_nbs<double>(p, j, i);
    p.rhsr[c] = rhs_sal(p, n, h, p.rusal[c], k);
    p.rusal[c] = h;
}

// ---------------------------------------------------------------------------
// wavefront tridiagonal solve (SolveImpEqnUpdate_{X,YZ,Temp,Sal})
// ---------------------------------------------------------------------------
// Inclusive scan of affine maps y -> A y + B across the 64 lanes, in lane
// order (UP) or reverse lane order.  Composition keeps the later map outside.
template <bool UP>
__device__ __forceinline__ void wave_affine_scan(double &A, double &B) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        double Ap = UP ? __shfl_up(A, off, 64) : __shfl_down(A, off, 64);
        double Bp = UP ? __shfl_up(B, off, 64) : __shfl_down(B, off, 64);
        bool ok = UP ? (lane >= off) : (lane + off < 64);
        if (ok) { B = A * Bp + B; A = A * Ap; }
    }
}

// Solve the normalised system on the CH rows a lane owns (v in: raw RHS d,
// v out: solution x), with factors f (see TriFactors).
template <int CH>
__device__ __forceinline__ void wave_tri_solve(double (&v)[CH], const TriFactors &f) {
    const int lane = threadIdx.x & 63;
    const double *l = f.l + lane * CH, *e = f.e + lane * CH, *g = f.g + lane * CH, *sc = f.s + lane * CH;
#pragma unroll
    for (int m = 0; m < CH; ++m) v[m] *= sc[m];
    // forward: y_r = v_r - l_r y_{r-1}
    double A = 1.0, B = 0.0;
#pragma unroll
    for (int m = 0; m < CH; ++m) { const double lm = l[m]; B = -lm * B + v[m]; A = -lm * A; }
    wave_affine_scan<true>(A, B);
    double y = __shfl_up(B, 1, 64);
    if (lane == 0) y = 0.0;
#pragma unroll
    for (int m = 0; m < CH; ++m) { y = -l[m] * y + v[m]; v[m] = y; }
    // backward: x_r = g_r y_r - e_r x_{r+1}
    A = 1.0; B = 0.0;
#pragma unroll
    for (int m = CH - 1; m >= 0; --m) { const double em = e[m]; B = -em * B + g[m] * v[m]; A = -em * A; }
    wave_affine_scan<false>(A, B);
    double x = __shfl_down(B, 1, 64);
    if (lane == 63) x = 0.0;
#pragma unroll
    for (int m = CH - 1; m >= 0; --m) { x = -e[m] * x + g[m] * v[m]; v[m] = x; }
}

// 2x2 projective matrix (normalised so its largest entry is 1)
struct Mob { double m00, m01, m10, m11; };
__device__ __forceinline__ Mob mob_mul(const Mob &x, const Mob &y) {   // x * y
    Mob r{x.m00 * y.m00 + x.m01 * y.m10, x.m00 * y.m01 + x.m01 * y.m11,
          x.m10 * y.m00 + x.m11 * y.m10, x.m10 * y.m01 + x.m11 * y.m11};
    const double mx = fmax(fmax(fabs(r.m00), fabs(r.m01)), fmax(fabs(r.m10), fabs(r.m11)));
    if (mx > 0.0) { const double q = 1.0 / mx; r.m00 *= q; r.m01 *= q; r.m10 *= q; r.m11 *= q; }
    return r;
}

// Solve a tridiagonal system whose rows differ from column to column (row
// r: a_r x_{r-1} + x_r + c_r x_{r+1} = v_r), CH rows per lane.  The Thomas
// recurrence c'_r = c_r / (1 - a_r c'_{r-1}) is a Moebius map of c'_{r-1};
// its prefix over the wavefront is a scan of 2x2 matrix products.  With c'
// known, forward elimination and back substitution are affine scans as in
// wave_tri_solve.
// c' of the row before this lane's first row: the Moebius prefix of the
// earlier lanes' rows applied to c' = 0
template <int CH>
__device__ __forceinline__ double wave_mobius_prefix(const double (&a)[CH], const double (&c)[CH]) {
    const int lane = threadIdx.x & 63;
    Mob L{1.0, 0.0, 0.0, 1.0};
#pragma unroll
    for (int m = 0; m < CH; ++m) L = mob_mul(Mob{0.0, c[m], -a[m], 1.0}, L);
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        Mob P{__shfl_up(L.m00, off, 64), __shfl_up(L.m01, off, 64), __shfl_up(L.m10, off, 64), __shfl_up(L.m11, off, 64)};
        if (lane >= off) L = mob_mul(L, P);
    }
    // the exclusive prefix applied to (0, 1)
    const double p0 = __shfl_up(L.m01, 1, 64), q0 = __shfl_up(L.m11, 1, 64);
    return lane == 0 ? 0.0 : p0 / q0;
}

template <int CH>
__device__ __forceinline__ void wave_tri_solve_general(double (&v)[CH], const double (&a)[CH], const double (&c)[CH]) {
    const int lane = threadIdx.x & 63;
    double t = wave_mobius_prefix<CH>(a, c);
    double cp[CH], g[CH];
#pragma unroll
    for (int m = 0; m < CH; ++m) { g[m] = 1.0 / (1.0 - a[m] * t); cp[m] = c[m] * g[m]; t = cp[m]; }
    // forward: y_r = g_r v_r - g_r a_r y_{r-1}
    double A = 1.0, B = 0.0;
#pragma unroll
    for (int m = 0; m < CH; ++m) { const double am = -g[m] * a[m]; B = am * B + g[m] * v[m]; A = am * A; }
    wave_affine_scan<true>(A, B);
    double y = __shfl_up(B, 1, 64);
    if (lane == 0) y = 0.0;
#pragma unroll
    for (int m = 0; m < CH; ++m) { y = -g[m] * a[m] * y + g[m] * v[m]; v[m] = y; }
    // backward: x_r = y_r - c'_r x_{r+1}
    A = 1.0; B = 0.0;
#pragma unroll
    for (int m = CH - 1; m >= 0; --m) { B = -cp[m] * B + v[m]; A = -cp[m] * A; }
    wave_affine_scan<false>(A, B);
    double x = __shfl_down(B, 1, 64);
    if (lane == 63) x = 0.0;
#pragma unroll
    for (int m = CH - 1; m >= 0; --m) { x = -cp[m] * x + v[m]; v[m] = x; }
}

// One column per wavefront: q[r] += solve(rhs)[r] for r in [u0,u1); rows
// listed in zero0/zero1 (if >= 0) are set to zero afterwards (the wall rows
// of vx, ImplicitAndUpdateVX.F90:86-87).  rhs holds the raw RHS on entry and
// the increment on exit when keep_rhs is set (as the reference's rhs array
// does); the fused step skips that write.
template <int CH>
__global__ void __launch_bounds__(256) k_tri_update(TriFactors f, double *rhs, double *q, int ldx,
                                                    long long plane, int ny, long long ncols, int u0, int u1,
                                                    int zero0, int zero1, int keep_rhs) {
    const long long col = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (col >= ncols) return;
    const int lane = threadIdx.x & 63;
    const int j = int(col % ny), i = int(col / ny);
    const long long base = (long long)i * plane + (long long)j * ldx;
    double v[CH];
#pragma unroll
    for (int m = 0; m < CH; ++m) {
        const int r = lane * CH + m;
        v[m] = r < f.n ? rhs[base + r] : 0.0;
    }
    wave_tri_solve<CH>(v, f);
#pragma unroll
    for (int m = 0; m < CH; ++m) {
        const int r = lane * CH + m;
        if (r < f.n) {
            if (keep_rhs) rhs[base + r] = v[m];
            if (r >= u0 && r < u1) q[base + r] += v[m];
            if (r == zero0 || r == zero1) q[base + r] = 0.0;
        }
    }
}

// ---------------------------------------------------------------------------
// fused column kernels: explicit terms + implicit RHS + tridiagonal solve +
// update of one wall-normal column per wavefront.  Stencil phase: lane l
// handles rows l, l+64, ... (coalesced loads of the column and its y/z
// neighbours); the RHS goes through LDS to the chunked layout of the scan
// solver and back.  Fields are read from the pre-substep arrays and the
// updated column is written to a second buffer (other wavefronts still read
// the old values as neighbours).
// ---------------------------------------------------------------------------
// Consecutive workgroups are dealt round-robin to the 8 XCDs; give each XCD
// a contiguous range of columns so y/z neighbours share its L2.
// The grid has a multiple of 8 workgroups (padded by the host); the map is a
// bijection of [0, gridDim.x) and indices >= the real count are idle.
__device__ __forceinline__ long long xcd_block(long long) {
    const long long b = blockIdx.x;
    const long long per = gridDim.x / 8;
    return (b % 8) * per + b / 8;
}
// A 1-D grid over n items, padded to a multiple of 8 workgroups.  Through
// xcd_block each XCD takes a contiguous range of them, so neighbours, which
// read the same halo cache lines, run on one L2 at about the same time.
__host__ __device__ __forceinline__ unsigned tile_grid(long long ntiles) { return unsigned((ntiles + 7) / 8 * 8); }
// Column walk: a workgroup owns 4 consecutive y columns, one per
// wavefront; workgroups form strips of STRIP_BLOCKS*4 columns in y, walked
// along z, so the y and z neighbour columns a wavefront reads belong to its
// own workgroup or to workgroups that ran just before it on the same XCD
// (still in its L2).
constexpr int STRIP_BLOCKS = 4;
__host__ __device__ __forceinline__ long long strip_blocks(int ny, int nz) {
    return (long long)((ny + 4 * STRIP_BLOCKS - 1) / (4 * STRIP_BLOCKS)) * STRIP_BLOCKS * nz;
}
// (j, i) of this wavefront's column; false if the slot is idle
__device__ __forceinline__ bool strip_column(long long blk, int wave, int ny, int nz, int &j, int &i) {
    const long long per_strip = (long long)STRIP_BLOCKS * nz;
    const long long strip = blk / per_strip, rem = blk % per_strip;
    i = int(rem / STRIP_BLOCKS);
    j = int(strip * 4 * STRIP_BLOCKS + (rem % STRIP_BLOCKS) * 4 + wave);
    const bool ok = blk < strip_blocks(ny, nz) && j < ny && i < nz;
    if (!ok) { j = 0; i = 0; }
    return ok;
}

// Row r of a column lives at lds_row<CH>(r): chunks of CH rows at an odd
// stride of CHP >= CH+1 doubles, so the solver's lane-strided 64-bit reads
// (lane * CHP) hit distinct bank pairs.
template <int CH>
constexpr int lds_chunk() { return (CH + 1) % 2 ? CH + 1 : CH + 2; }
// Tight form: CH itself when odd (lane strides of 2*CH dwords reach 16
// distinct bank pairs per 16 lanes), else CH+1.
template <int CH>
constexpr int lds_chunk_tight() { return CH % 2 ? CH : CH + 1; }
template <int CH, int CHP = lds_chunk<CH>()>
__device__ __forceinline__ unsigned lds_row(unsigned r) { return (r / CH) * CHP + r % CH; }
template <int CH, int CHP = lds_chunk<CH>()>
constexpr int lds_col_size() { return 64 * CHP; }

template <int CH, int CHP = lds_chunk<CH>()>
__device__ __forceinline__ void column_solve_lds(double *buf, const TriFactors &f) {
    const int lane = threadIdx.x & 63;
    double v[CH];
#pragma unroll
    for (int m = 0; m < CH; ++m) v[m] = buf[lane * CHP + m];
    wave_tri_solve<CH>(v, f);
#pragma unroll
    for (int m = 0; m < CH; ++m) buf[lane * CHP + m] = v[m];
}

// Masked solve of one column held in LDS (SolveImpEqnUpdate_X_pf /
// _YZ_pf, phasefield.F90:821-930): rows flagged in msk are the identity with
// the right-hand side already in buf; the others are the rows of f.
template <int CH>
__device__ __forceinline__ void column_solve_masked_lds(double *buf, const double *msk, const TriFactors &f) {
    const int lane = threadIdx.x & 63;
    double v[CH], a[CH], c[CH];
#pragma unroll
    for (int m = 0; m < CH; ++m) {
        const int r = lane * CH + m;
        const bool solid = msk[lane * lds_chunk<CH>() + m] != 0.0;
        const double sv = f.s[r];
        v[m] = buf[lane * lds_chunk<CH>() + m];
        if (!solid) v[m] *= sv;
        a[m] = solid ? 0.0 : f.a[r];
        c[m] = solid ? 0.0 : f.c[r];
    }
    wave_tri_solve_general<CH>(v, a, c);
#pragma unroll
    for (int m = 0; m < CH; ++m) buf[lane * lds_chunk<CH>() + m] = v[m];
}

// two-element vector of the storage type (64-bit or 128-bit lane accesses)
template <typename RT> struct Pair;
template <> struct Pair<float> { using T = float2; };
template <> struct Pair<double> { using T = double2; };
// Explicit terms of vx, vy, vz, T (+ AddSalBuoyancy) and ImplicitAndUpdate
// VX/VY/VZ/Temp with their solves (TimeMarcher.F90:45-95) for one column.
struct BaseOut { double *vx, *vy, *vz, *temp; };

// stencil phase of field FLD: RHS of each row into buf, old value into own.
// HT is the storage and arithmetic type of the explicit terms (and of salc);
// the RHS and the solve run in FP64.  With PF (phase field) the velocity
// terms lose the volume penalty (AddVolumePenalty, phasefield.F90:525-566),
// the temperature term gains the latent heat qlat (AddLatentHeat, :651-725),
// and a velocity row whose averaged phic exceeds pf_direct_force = 0.9
// (phasefield.F90:29) is flagged in msk with right-hand side -u, the
// identity row of SolveImpEqnUpdate_X_pf / _YZ_pf (:821-930).
template <int FLD, int CH, typename HT, bool PF>
__device__ __forceinline__ void column_base_rows(const KP &p, const Nb &n, long long c0, double *buf, double *own,
                                                 double *msk, unsigned lane, unsigned nrow, bool live) {
    const HT *salc = sel<HT>(p.salc, p.salcf) + c0;
    HT *ru = (FLD == 0 ? sel<HT>(p.rux, p.ruxf) : FLD == 1 ? sel<HT>(p.ruy, p.ruyf)
              : FLD == 2 ? sel<HT>(p.ruz, p.ruzf) : sel<HT>(p.rut, p.rutf)) + c0;
    const unsigned nxm = p.nxm;
#pragma unroll 1
    for (unsigned r = lane; r < nrow; r += 64) {
        double rhs = 0.0, old = 0.0;
        bool solid = false;
        if (live && r < unsigned(p.nx)) {
            const HT sb = (p.active_s == 1 && r < nxm) ? HT(p.bycs) * salc[r] : HT(0);
            if (FLD == 0) {
                old = n.vx[r];
                if (r >= 1 && r < nxm) {
                    HT h;
                    double bref = 0.0;
                    if (sizeof(HT) == sizeof(float) && p.bref) {
                        // FP32 terms: the buoyancy enters as its deviation from
                        // the row's FP64 reference, formed in FP64 and rounded
                        // once; the RHS adds the reference back in FP64
                        bref = p.bref[r];
                        h = ex_vx<HT, false>(p, n, r) + HT(p.byct * (p.active_t * 0.5 * (n.t[r] + n.t[r - 1])) - bref);
                    } else {
                        h = ex_vx<HT>(p, n, r);
                    }
                    if (p.gaxis == 1) h -= sb;
                    if (PF) {
                        h -= HT((n.pc[r] + n.pc[r - 1]) * n.vx[r] * p.heta);
                        solid = 0.5 * (n.pc[r] + n.pc[r + 1]) > 0.9;
                    }
                    rhs = rhs_vx(p, n, double(h) + bref, double(ru[r]) + bref, r);
                    ru[r] = h;
                } else if (PF) {
                    solid = true;                    // rows 1 and nx: identity with rhs -vx
                }
            } else if (FLD == 1) {
                old = n.vy[r];
                if (r < nxm) {
                    HT h = ex_vy<HT>(p, n, r);
                    if (p.gaxis == 2) h -= sb;
                    if (PF) {
                        const double pa = n.pc[r] + n.pc_jm[r];
                        h -= HT(pa * n.vy[r] * p.heta);
                        solid = 0.5 * pa > 0.9;
                    }
                    rhs = rhs_vy(p, n, double(h), double(ru[r]), r);
                    ru[r] = h;
                }
            } else if (FLD == 2) {
                old = n.vz[r];
                if (r < nxm) {
                    HT h = ex_vz<HT>(p, n, r);
                    if (p.gaxis == 3) h -= sb;
                    if (PF) {
                        const double pa = n.pc[r] + n.pc_im[r];
                        h -= HT(pa * n.vz[r] * p.heta);
                        solid = 0.5 * pa > 0.9;
                    }
                    rhs = rhs_vz(p, n, double(h), double(ru[r]), r);
                    ru[r] = h;
                }
            } else {
                old = n.t[r];
                if (r < nxm) {
                    HT h = ex_temp<HT>(p, n, r);
                    if (PF) h += HT(p.qlat[c0 + r]);
                    if (p.moist) h = HT(double(h) + condensation_heat(p, c0, r));
                    rhs = rhs_temp(p, n, double(h), double(ru[r]), r);
                    ru[r] = h;
                }
            }
        }
        if (PF && FLD < 3) {
            if (solid) rhs = -old;
            msk[lds_row<CH>(r)] = solid ? 1.0 : 0.0;
        }
        buf[lds_row<CH>(r)] = rhs;
        own[lds_row<CH>(r)] = old;
    }
}

// Four passes, one field each (the phase-field form, and wall-normal sizes
// above 512 cells).  CH = ceil(nx / 64).
template <int CH, typename HT, bool PF>
__global__ void __launch_bounds__(256) k_column_base(KP p, TriFactors fx, TriFactors fyz, TriFactors ft, BaseOut o) {
    __shared__ double lds[PF ? 3 : 2][4][lds_col_size<CH>()];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned lane = threadIdx.x & 63;
    int j, i;
    const bool live = strip_column(xcd_block(0), wave, p.ny, p.nz, j, i);
    double *buf = lds[0][wave], *own = lds[1][wave], *msk = lds[PF ? 2 : 1][wave];
    const Nb n = make_nb(p, j, i);
    const long long c0 = (long long)i * p.plane + (long long)j * p.ldx;
    const unsigned nrow = 64 * CH, nx = p.nx, nxm = p.nxm;
#pragma unroll 1
    for (int fld = 0; fld < 4; ++fld) {
        switch (fld) {
        case 0: column_base_rows<0, CH, HT, PF>(p, n, c0, buf, own, msk, lane, nrow, live); break;
        case 1: column_base_rows<1, CH, HT, PF>(p, n, c0, buf, own, msk, lane, nrow, live); break;
        case 2: column_base_rows<2, CH, HT, PF>(p, n, c0, buf, own, msk, lane, nrow, live); break;
        default: column_base_rows<3, CH, HT, PF>(p, n, c0, buf, own, msk, lane, nrow, live); break;
        }
        __syncthreads();
        const TriFactors &f = fld == 0 ? fx : (fld == 3 ? ft : fyz);
        if (PF && fld < 3) column_solve_masked_lds<CH>(buf, msk, f);
        else column_solve_lds<CH>(buf, f);
        __syncthreads();
        if (live) {
            double *out = (fld == 0 ? o.vx : fld == 1 ? o.vy : fld == 2 ? o.vz : o.temp) + c0;
            for (unsigned r = lane; r < nx; r += 64) {
                const unsigned q = lds_row<CH>(r);
                double v = own[q];
                if (fld == 0) v = (r >= 1 && r < nxm) ? v + buf[q] : 0.0;   // walls, ImplicitAndUpdateVX.F90:86-87
                else if (r < nxm) v += buf[q];
                out[r] = v;
            }
        }
        __syncthreads();
    }
}

// Right-hand sides of vx, vy, vz and T at row r < nx of one column (the
// stencil phase of column_base_rows for the four fields at once, with the phase
// field): every neighbour value is loaded once for the four explicit terms,
// and the explicit terms are stored to their history arrays after all
// loads.  Rows without an equation (vx rows 0 and nxm, the unused index
// nxm of the others) give 0.
template <typename HT>
__device__ __forceinline__ void base_rhs4(const KP &p, const Nb &n, long long c0, unsigned r, double (&rhs)[4],
                                          unsigned &solid) {
    const unsigned nxm = p.nxm;
    HT *rux = sel<HT>(p.rux, p.ruxf) + c0, *ruy = sel<HT>(p.ruy, p.ruyf) + c0;
    HT *ruz = sel<HT>(p.ruz, p.ruzf) + c0, *rut = sel<HT>(p.rut, p.rutf) + c0;
    const bool wx = r >= 1 && r < nxm, wc = r < nxm;
    const HT sb = (p.active_s == 1 && wc) ? HT(p.bycs) * sel<HT>(p.salc, p.salcf)[c0 + r] : HT(0);
    HT h0 = HT(0), h1 = HT(0), h2 = HT(0), h3 = HT(0);
    double bref = 0.0, r0 = 0.0, r1 = 0.0, r2 = 0.0, r3 = 0.0;
    // phase field: solid rows of vx, vy, vz (bits 0..2); vx rows 0 and nxm
    // are identity rows (SolveImpEqnUpdate_X_pf)
    bool sx = !wx, sy = false, sz = false;
    if (wx) {
        if (sizeof(HT) == sizeof(float) && p.bref) {
            // FP32 terms: buoyancy as its deviation from the row's FP64
            // reference, which the RHS adds back in FP64
            bref = p.bref[r];
            h0 = ex_vx<HT, false>(p, n, r) + HT(p.byct * (p.active_t * 0.5 * (n.t[r] + n.t[r - 1])) - bref);
        } else {
            h0 = ex_vx<HT>(p, n, r);
        }
        if (p.gaxis == 1) h0 -= sb;
        // AddVolumePenalty (phasefield.F90:525-566); the row is solid where
        // the averaged phic exceeds pf_direct_force = 0.9 (:29, :821-930)
        h0 -= HT((n.pc[r] + n.pc[r - 1]) * n.vx[r] * p.heta);
        sx = 0.5 * (n.pc[r] + n.pc[r + 1]) > 0.9;
        r0 = double(rux[r]);
    }
    if (wc) {
        h1 = ex_vy<HT>(p, n, r);
        if (p.gaxis == 2) h1 -= sb;
        h2 = ex_vz<HT>(p, n, r);
        if (p.gaxis == 3) h2 -= sb;
        h3 = ex_temp<HT>(p, n, r);
        const double py = n.pc[r] + n.pc_jm[r], pz = n.pc[r] + n.pc_im[r];
        h1 -= HT(py * n.vy[r] * p.heta);
        h2 -= HT(pz * n.vz[r] * p.heta);
        sy = 0.5 * py > 0.9;
        sz = 0.5 * pz > 0.9;
        h3 += HT(p.qlat[c0 + r]);                // AddLatentHeat (:651-725)
        if (p.moist) h3 = HT(double(h3) + condensation_heat(p, c0, r));
        r1 = double(ruy[r]); r2 = double(ruz[r]); r3 = double(rut[r]);
    }
    rhs[0] = wx ? rhs_vx(p, n, double(h0) + bref, r0 + bref, r) : 0.0;
    rhs[1] = wc ? rhs_vy(p, n, double(h1), r1, r) : 0.0;
    rhs[2] = wc ? rhs_vz(p, n, double(h2), r2, r) : 0.0;
    rhs[3] = wc ? rhs_temp(p, n, double(h3), r3, r) : 0.0;
    // a solid row is the identity with right-hand side -u
    if (sx) rhs[0] = -n.vx[r];
    if (sy) rhs[1] = -n.vy[r];
    if (sz) rhs[2] = -n.vz[r];
    solid = unsigned(sx) | unsigned(sy) << 1 | unsigned(sz) << 2;
    if (wx) rux[r] = h0;
    if (wc) { ruy[r] = h1; ruz[r] = h2; rut[r] = h3; }
}

// Masked solve of one column in LDS (tight layout CHP) with the solid flags
// of its rows as bytes in natural row order (mskb[r] != 0: identity row,
// right-hand side already in buf); the other rows are those of f
template <int CH, int CHP>
__device__ __forceinline__ void column_solve_masked_bytes(double *buf, const unsigned char *mskb, const TriFactors &f) {
    const int lane = threadIdx.x & 63;
    double v[CH], a[CH], c[CH];
#pragma unroll
    for (int m = 0; m < CH; ++m) {
        const int r = lane * CH + m;
        const bool solid = mskb[r] != 0;
        v[m] = buf[lane * CHP + m];
        if (!solid) v[m] *= f.s[r];
        a[m] = solid ? 0.0 : f.a[r];
        c[m] = solid ? 0.0 : f.c[r];
    }
    wave_tri_solve_general<CH>(v, a, c);
#pragma unroll
    for (int m = 0; m < CH; ++m) buf[lane * CHP + m] = v[m];
}

// Single-pass form of k_column_base with the phase field.  One sweep over the rows forms the
// four right-hand sides, loading every neighbour value once for all four
// explicit terms.  Those of vx and vy go to two LDS columns of the
// wavefront, those of vz and T stay in registers.  The vx and vy solves and
// updates follow, then the vz and T right-hand sides move into the same two
// LDS columns for their solves and updates.  Two LDS columns per wavefront
// instead of four keep 4 wavefronts per SIMD; the updates read the old value
// of the own column again (from cache).
// The velocity terms carry the volume penalty, T the latent heat,
// and solid velocity rows are identity rows: their flags go to LDS as bytes
// (vx, vy; vz's flags wait in a register bit mask) for the masked solves.
// CH = ceil(nxm / 64) is the size of the largest system (nxm rows); when
// nx = 64 CH + 1 the last face has no equation (the wall of vx, the unused
// index of the others) and only the update touches it.
template <int CH, typename HT>
__global__ void __launch_bounds__(256) k_column_base1(KP p, TriFactors fx, TriFactors fyz, TriFactors ft, BaseOut o) {
    constexpr int CHP = lds_chunk_tight<CH>();
    constexpr unsigned NROW = 64u * CH;
    __shared__ double lds[4][2][lds_col_size<CH, CHP>()];
    __shared__ unsigned char mskb[4][2][NROW];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned lane = threadIdx.x & 63;
    int j, i;
    const bool live = strip_column(xcd_block(0), wave, p.ny, p.nz, j, i);
    const Nb n = make_nb(p, j, i);
    const long long c0 = (long long)i * p.plane + (long long)j * p.ldx;
    const unsigned nx = p.nx, nxm = p.nxm;
    double *b0 = lds[wave][0], *b1 = lds[wave][1];
    unsigned char *m0 = mskb[wave][0], *m1 = mskb[wave][1];
    double keep[2][CH];                          // right-hand sides of vz and T
    unsigned zsolid = 0;                         // vz's solid flags, bit m for row lane + 64 m
#pragma unroll
    for (int m = 0; m < CH; ++m) {
        const unsigned r = lane + 64u * m;
        double rhs[4] = {0.0, 0.0, 0.0, 0.0};
        unsigned solid = 0;
        if (live && r < nxm) base_rhs4<HT>(p, n, c0, r, rhs, solid);
        const unsigned q = lds_row<CH, CHP>(r);
        b0[q] = rhs[0];
        b1[q] = rhs[1];
        keep[0][m] = rhs[2];
        keep[1][m] = rhs[3];
        m0[r] = (unsigned char)(solid & 1u);
        m1[r] = (unsigned char)((solid >> 1) & 1u);
        zsolid |= ((solid >> 2) & 1u) << m;
    }
    __syncthreads();
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        if (g == 1) {
#pragma unroll
            for (int m = 0; m < CH; ++m) {
                const unsigned q = lds_row<CH, CHP>(lane + 64u * m);
                b0[q] = keep[0][m];
                b1[q] = keep[1][m];
                m0[lane + 64u * m] = (unsigned char)((zsolid >> m) & 1u);
            }
            __syncthreads();
        }
        column_solve_masked_bytes<CH, CHP>(b0, m0, g == 0 ? fx : fyz);
        if (g == 0) column_solve_masked_bytes<CH, CHP>(b1, m1, fyz);
        else column_solve_lds<CH, CHP>(b1, ft);
        __syncthreads();
        if (live) {
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                const int fld = 2 * g + f;
                const double *old = fld == 0 ? n.vx : fld == 1 ? n.vy : fld == 2 ? n.vz : n.t;
                double *out = (fld == 0 ? o.vx : fld == 1 ? o.vy : fld == 2 ? o.vz : o.temp) + c0;
                const double *d = f == 0 ? b0 : b1;
#pragma unroll 1
                for (unsigned r = lane; r < nx; r += 64) {
                    const double u = old[r];
                    const double x = d[lds_row<CH, CHP>(r < NROW ? r : NROW - 1)];
                    if (fld == 0) out[r] = (r >= 1 && r < nxm) ? u + x : 0.0;     // walls, ImplicitAndUpdateVX.F90:86-87
                    else out[r] = r < nxm ? u + x : u;
                }
            }
        }
        if (g == 0) __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// pressure projection point kernels
// ---------------------------------------------------------------------------
// CalcLocalDivergence, pressure.F90:147-161
__global__ void __launch_bounds__(256) k_local_divergence(KP p) {
    AFID_POINT_PROLOGUE(p.nxm, p.ny, p.nz)
    const double usdtal = 1.0 / (p.dt * p.al);
    const double dq = (p.vz[bidx(p, k, j, ip)] - p.vz[bidx(p, k, j, i)]) * p.dz
                    + (p.vy[bidx(p, k, jp, i)] - p.vy[bidx(p, k, j, i)]) * p.dy
                    + (p.vx[bidx(p, k + 1, j, i)] - p.vx[bidx(p, k, j, i)]) * p.udx3m[k];
    p.dph[bidx(p, k, j, i)] = dq * usdtal;
}

// RemoveDivergence (pressure.F90:245-266) and/or CorrectPressure
// (pressure.F90:276-300); both read only dph, so one sweep does both.
// DT: storage type of dph (FP32 in the mixed form's sweeps)
template <typename DT>
__global__ void __launch_bounds__(256) k_project(KP p, int do_vel, int do_pr, Gate gate) {
    if (gate_closed(gate)) return;
    const int k = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y;
    if (k >= p.nxm || j >= p.ny) return;
    const int jm = wrapm(j, p.ny), jp = wrapp(j, p.ny);
    const DT *d = sel<DT>(p.dph, p.dphf);
    const int km = k == 0 ? 0 : k - 1, kp = k == p.nxm - 1 ? k : k + 1;
    // z walked with the grid's z stride: a full grid (one plane each) or, for
    // a gated launch, a short grid that costs little when the gate is closed
    // every load of a cell ahead of its stores (the fields may alias as far
    // as the compiler knows; interleaved stores would serialise the loads)
    for (int i = blockIdx.z; i < p.nz; i += gridDim.z) {
        const int im = wrapm(i, p.nz), ip = wrapp(i, p.nz);
        const long long c = bidx(p, k, j, i);
        const double dc = d[c], dkm = d[bidx(p, km, j, i)], djm = d[bidx(p, k, jm, i)], dim = d[bidx(p, k, j, im)];
        if (do_vel) {
            const double adt = p.al * p.dt;
            const double ux = p.vx[c], uy = p.vy[c], uz = p.vz[c];
            const double nux = ux - (dc - dkm) * (adt * p.udx3c[k]);
            const double nuy = uy - (dc - djm) * (adt * p.dy);
            const double nuz = uz - (dc - dim) * (adt * p.dz);
            if (do_pr) {
                const double be = p.al * p.beta, prc = p.pr[c];
                const double npr = prc + (dc - be * ((d[bidx(p, k, j, ip)] - 2.0 * dc + dim) * p.dzq +
                                                     (d[bidx(p, k, jp, i)] - 2.0 * dc + djm) * p.dyq +
                                                     (d[bidx(p, kp, j, i)] * p.apphk[k] + dc * p.acphk[k] + dkm * p.amphk[k])));
                p.pr[c] = npr;
            }
            p.vx[c] = nux; p.vy[c] = nuy; p.vz[c] = nuz;
        } else if (do_pr) {
            const double be = p.al * p.beta;
            p.pr[c] += dc - be * ((d[bidx(p, k, j, ip)] - 2.0 * dc + dim) * p.dzq +
                                  (d[bidx(p, k, jp, i)] - 2.0 * dc + djm) * p.dyq +
                                  (d[bidx(p, kp, j, i)] * p.apphk[k] + dc * p.acphk[k] + dkm * p.amphk[k]));
        }
    }
}

// The same projection writing the corrected velocity to a second buffer
// (u_out), so that every cell can also form the divergence the corrected
// field will have (its own and its +1 neighbours' faces, from the old
// velocity and dph): the FP64 residual of the mixed form's iterative
// refinement, max-reduced into *slot (CheckDivergence units).  Each thread
// marches along z over PROJ_ZC planes and carries dph and vz of the planes
// i-1, i, i+1 in registers, so no plane is read twice.  A workgroup's maximum
// goes straight to the slot: 32 768 of them cost nothing at 256 x 512^2 (project
// 3672 us a step; with partial maxima and a kernel over them 3690), and at 64^3
// the second launch was 5 us of every substep.
constexpr int PROJ_ZC = 8;
__global__ void __launch_bounds__(256) k_project_res(KP p, double *vx_out, double *vy_out, double *vz_out,
                                                     unsigned long long *slot) {
    const int k = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y;
    const int i0 = blockIdx.z * PROJ_ZC, i1 = min(i0 + PROJ_ZC, p.nz);
    double dvm = 0.0;
    if (k < p.nxm && j < p.ny) {
        const int jm = wrapm(j, p.ny), jp = wrapp(j, p.ny);
        const int km = k == 0 ? 0 : k - 1, kp = k == p.nxm - 1 ? k : k + 1;
        const float *d = p.dphf;                  // the mixed form's FP32 sweep correction
        const double adt = p.al * p.dt, be = p.al * p.beta;
        const double ucx = adt * p.udx3c[k], ucx1 = k + 1 <= p.nxm - 1 ? adt * p.udx3c[k + 1] : 0.0;
        const long long row = (long long)j * p.ldx + k, rowjm = (long long)jm * p.ldx + k, rowjp = (long long)jp * p.ldx + k;
        double d_m = d[(long long)wrapm(i0, p.nz) * p.plane + row];
        double d_c = d[(long long)i0 * p.plane + row];
        double w_c = p.vz[(long long)i0 * p.plane + row];
        for (int i = i0; i < i1; ++i) {
            const long long pl = (long long)i * p.plane, plp = (long long)wrapp(i, p.nz) * p.plane;
            const long long c = pl + row;
            // every load of the cell ahead of its stores (the outputs may
            // alias the inputs as far as the compiler knows)
            const double d_p = d[plp + row], w_p = p.vz[plp + row];
            const double dkm = d[pl + row - k + km], dkp = d[pl + row - k + kp];
            const double djm = d[pl + rowjm], djp = d[pl + rowjp];
            const double vxc = p.vx[c], vyc = p.vy[c], vx1 = p.vx[c + 1], vy1 = p.vy[pl + rowjp];
            const double d1 = d[c + 1], prc = p.pr[c];
            // corrected faces of this cell (as k_project)
            const double ux = vxc - (d_c - dkm) * ucx;
            const double uy = vyc - (d_c - djm) * (adt * p.dy);
            const double uz = w_c - (d_c - d_m) * (adt * p.dz);
            // corrected +1 faces (owned by the neighbouring cells)
            const double ux1 = k + 1 <= p.nxm - 1 ? vx1 - (d1 - d_c) * ucx1 : vx1;
            const double uy1 = vy1 - (djp - d_c) * (adt * p.dy);
            const double uz1 = w_p - (d_p - d_c) * (adt * p.dz);
            dvm = fmax(dvm, fabs((uz1 - uz) * p.dz + (uy1 - uy) * p.dy + (ux1 - ux) * p.udx3m[k]));
            const double npr = prc + (d_c - be * ((d_p - 2.0 * d_c + d_m) * p.dzq + (djp - 2.0 * d_c + djm) * p.dyq +
                                                 (dkp * p.apphk[k] + d_c * p.acphk[k] + dkm * p.amphk[k])));
            if (k == p.nxm - 1) {      // index nx: wall face of vx (not corrected), unused for vy, vz
                const double wy = p.vy[c + 1], wz = p.vz[c + 1];
                vx_out[c + 1] = vx1; vy_out[c + 1] = wy; vz_out[c + 1] = wz;
            }
            vx_out[c] = ux; vy_out[c] = uy; vz_out[c] = uz;
            p.pr[c] = npr;
            d_m = d_c; d_c = d_p; w_c = w_p;
        }
    }
    max_to_slot(slot, block_max(dvm));
}

// ---------------------------------------------------------------------------
// multiresolution transfers
// ---------------------------------------------------------------------------
// periodic wrap of an index a few periods away at most, without a division
__device__ __forceinline__ int wrapf(int j, int n) {
    while (j < 0) j += n;
    while (j >= n) j -= n;
    return j;
}

// Inclusive prefix sum over the 64 lanes of a wavefront with DPP lane
// moves: Kogge-Stone within each row of 16 lanes (row_shr 1, 2, 4, 8),
// then the row totals carried forward (row_bcast 15 into rows 1 and 3,
// row_bcast 31 into rows 2 and 3).  No LDS traffic.
template <int CTRL, int ROWS, bool BC>
__device__ __forceinline__ int dpp32(int v) { return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, BC); }
template <int CTRL, int ROWS, bool BC>
__device__ __forceinline__ float dpp_move(float v) { return __builtin_bit_cast(float, dpp32<CTRL, ROWS, BC>(__builtin_bit_cast(int, v))); }
template <int CTRL, int ROWS, bool BC>
__device__ __forceinline__ double dpp_move(double v) {
    const long long b = __builtin_bit_cast(long long, v);
    const int lo = dpp32<CTRL, ROWS, BC>(int(b & 0xffffffffLL)), hi = dpp32<CTRL, ROWS, BC>(int(b >> 32));
    return __builtin_bit_cast(double, (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
// value of lane 63 (the wavefront total of an inclusive scan), uniform
__device__ __forceinline__ float wave_lane63(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
__device__ __forceinline__ double wave_lane63(double v) {
    const long long b = __builtin_bit_cast(long long, v);
    const int lo = __builtin_amdgcn_readlane(int(b & 0xffffffffLL), 63), hi = __builtin_amdgcn_readlane(int(b >> 32), 63);
    return __builtin_bit_cast(double, (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
template <typename T>
__device__ __forceinline__ T wave_incl_scan(T v) {
    v += dpp_move<0x111, 0xf, true>(v);      // row_shr:1
    v += dpp_move<0x112, 0xf, true>(v);      // row_shr:2
    v += dpp_move<0x114, 0xf, true>(v);      // row_shr:4
    v += dpp_move<0x118, 0xf, true>(v);      // row_shr:8
    v += dpp_move<0x142, 0xa, false>(v);     // row_bcast:15
    v += dpp_move<0x143, 0xc, false>(v);     // row_bcast:31
    return v;
}

// ---------------------------------------------------------------------------
// seeded initial condition (CreateInitialConditions.F90:175-201 RBC branch)
// ---------------------------------------------------------------------------
__device__ __forceinline__ double splitmix_uniform(unsigned long long seed, unsigned long long idx) {
    unsigned long long z = (idx ^ seed) + 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z = z ^ (z >> 31);
    return double(z >> 11) * (1.0 / 9007199254740992.0);
}
// scalar = bottom + (top - bottom) x/alx3 + noise, noise amplitude clamped near
// the walls as the reference does (CreateInitialConditions.F90:187-201); the
// noise of point (k,j,i) is U[0,1) of splitmix64(seed ^ linear index) over the
// (nxf, ny, nz) array, x fastest.
template <typename FT>
__global__ void __launch_bounds__(256) k_init_scalar(FT *f, const double *bot, const double *top, const double *xm,
                                                     int nxm, int nxf, int ldx, int ny, int nz, double alx3,
                                                     double eps, unsigned long long seed) {
    const int k = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y, i = blockIdx.z;
    if (k >= nxf || j >= ny) return;
    const long long o = ((long long)i * ny + j) * ldx + k;
    if (k >= nxm) { f[o] = FT(0); return; }
    const long long p2 = (long long)i * ny + j;
    const double x = xm[k];
    double v = bot[p2] + (top[p2] - bot[p2]) * x / alx3;
    const double r = splitmix_uniform(seed, (unsigned long long)(((long long)i * ny + j) * nxf + k));
    const double amp = (fabs(x - 0.5) + eps > 0.5) ? 0.5 - fabs(x - 0.5) : eps;
    f[o] = FT(v + amp * (2.0 * r - 1.0));
}

// ---------------------------------------------------------------------------
// reductions
// ---------------------------------------------------------------------------
// CalcMaxCFL.F90:24-44 (what=0) / CheckDivergence.F90:24-43 (what=1) on the
// base grid, slot 0; refined grid versions write slot 1.
__global__ void __launch_bounds__(256) k_cfl_div(KP p, int what) {
    const int k = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y;
    double v = 0.0;
    for (int i = blockIdx.z; i < p.nz; i += gridDim.z) {
    if (k < p.nxm && j < p.ny) {
        const int jp = wrapp(j, p.ny), ip = wrapp(i, p.nz);
        double w;
        if (what == 0)
            w = fabs((p.vz[bidx(p, k, j, i)] + p.vz[bidx(p, k, j, ip)]) * 0.5 * p.dz)
              + fabs((p.vy[bidx(p, k, j, i)] + p.vy[bidx(p, k, jp, i)]) * 0.5 * p.dy)
              + fabs((p.vx[bidx(p, k, j, i)] + p.vx[bidx(p, k + 1, j, i)]) * 0.5 * p.udx3m[k]);
        else
            w = fabs((p.vz[bidx(p, k, j, ip)] - p.vz[bidx(p, k, j, i)]) * p.dz
                   + (p.vy[bidx(p, k, jp, i)] - p.vy[bidx(p, k, j, i)]) * p.dy
                   + (p.vx[bidx(p, k + 1, j, i)] - p.vx[bidx(p, k, j, i)]) * p.udx3m[k]);
        v = fmax(v, w);
    }
    }
    v = block_max(v);
    if (threadIdx.x == 0 && threadIdx.y == 0) atomicMax(&p.redmax[2 * what], (unsigned long long)__double_as_longlong(v));
}
template <typename RT>
__global__ void __launch_bounds__(256) k_cfl_div_r(KP p, int what) {
    const int k = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y;
    const RT *vxr = sel<RT>(p.vxr, p.vxrf), *vyr = sel<RT>(p.vyr, p.vyrf), *vzr = sel<RT>(p.vzr, p.vzrf);
    double v = 0.0;
    for (int i = blockIdx.z; i < p.nzr; i += gridDim.z) {
    if (k < p.nxmr && j < p.nyr) {
        const int jp = wrapp(j, p.nyr), ip = wrapp(i, p.nzr);
        double w;
        if (what == 0)
            w = fabs((double(vzr[ridx(p, k, j, i)]) + double(vzr[ridx(p, k, j, ip)])) * 0.5 * p.dzr)
              + fabs((double(vyr[ridx(p, k, j, i)]) + double(vyr[ridx(p, k, jp, i)])) * 0.5 * p.dyr)
              + fabs((double(vxr[ridx(p, k, j, i)]) + double(vxr[ridx(p, k + 1, j, i)])) * 0.5 * p.udx3mr[k]);
        else
            w = fabs((double(vzr[ridx(p, k, j, ip)]) - double(vzr[ridx(p, k, j, i)])) * p.dzr
                   + (double(vyr[ridx(p, k, jp, i)]) - double(vyr[ridx(p, k, j, i)])) * p.dyr
                   + (double(vxr[ridx(p, k + 1, j, i)]) - double(vxr[ridx(p, k, j, i)])) * p.udx3mr[k]);
        v = fmax(v, w);
    }
    }
    v = block_max(v);
    if (threadIdx.x == 0 && threadIdx.y == 0) atomicMax(&p.redmax[2 * what + 1], (unsigned long long)__double_as_longlong(v));
}

// GlobalQuantities.F90:39-60 partial sums per block: {T vxcen g3rc, T g3rc, (u^2+v^2+w^2) g3rc}
__global__ void __launch_bounds__(256) k_global_sums(KP p) {
    const int k = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y, i = blockIdx.z;
    double a = 0.0, b = 0.0, c = 0.0;
    if (k < p.nxm && j < p.ny) {
        const long long o = bidx(p, k, j, i);
        const double fac2 = p.g3rc[k];
        const double vxcen = (p.vx[o] + p.vx[o + 1]) * 0.5, t = p.temp[o];
        a = t * vxcen * fac2;
        b = t * fac2;
        c = fac2 * (p.vz[o] * p.vz[o] + p.vy[o] * p.vy[o] + p.vx[o] * p.vx[o]);
    }
    a = block_sum(a); b = block_sum(b); c = block_sum(c);
    if (threadIdx.x == 0 && threadIdx.y == 0) {
        const long long blk = ((long long)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
        p.redsum[3 * blk + 0] = a; p.redsum[3 * blk + 1] = b; p.redsum[3 * blk + 2] = c;
    }
}
__global__ void __launch_bounds__(256) k_sum_partials(const double *part, long long nblk, double *out) {
    double a = 0.0, b = 0.0, c = 0.0;
    for (long long q = threadIdx.x; q < nblk; q += blockDim.x) { a += part[3 * q]; b += part[3 * q + 1]; c += part[3 * q + 2]; }
    a = block_sum(a); b = block_sum(b); c = block_sum(c);
    if (threadIdx.x == 0) { out[0] = a; out[1] = b; out[2] = c; }
}

}  // namespace afid
