// afid_phase.hpp -- phase-field kernels (src/phasefield.F90): the explicit
// and implicit phi terms, the volume penalty and the masked velocity solves of
// the per-routine calls, and the seeded sphere.  In the fused step the phi
// column is k_column_refined and the masked solves are part of k_column_base1
// (four passes: k_column_base); the transfers (tempr, phic, latent heat) are in
// afid_transfer.hpp.
#pragma once
#include <hip/hip_runtime.h>
#include "afid_params.hpp"
#include "afid_stencils.hpp"
#include "afid_kernels.hpp"

namespace afid {

// ExplicitPhase, phasefield.F90:345-383, row k of a refined column: lateral
// diffusion D (phi_yy + phi_zz) minus the Allen-Cahn source
// pf_B phi (1 - phi) (1 - 2 phi + A (T_r - T_m)), in arithmetic T
template <typename T>
__device__ __forceinline__ T ex_phase_val(const KP &p, T pc, T pym, T pyp, T pzm, T pzp, T tr) {
    const T dyyp = (pyp - T(2.0) * pc + pym) * T(p.pf_d * p.dyqr);
    const T dzzp = (pzp - T(2.0) * pc + pzm) * T(p.pf_d * p.dzqr);
    const T nlphi = T(p.pf_b) * pc * (T(1.0) - pc) * (T(1.0) - T(2.0) * pc + T(p.pf_a) * (tr - T(p.pf_tm)));
    return dyyp + dzzp - nlphi;
}
// ImplicitPhase, phasefield.F90:386-419: zero-gradient x second derivative
__device__ __forceinline__ double rhs_phase_val(const KP &p, unsigned k, double h, double ru, double pm, double pc,
                                                double pp) {
    double dxxp;
    if (k == 0) dxxp = pp * p.ap3spkr[k] + pc * p.ac3spkr[k];
    else if (k == unsigned(p.nxmr - 1)) dxxp = pc * p.ac3spkr[k] + pm * p.am3spkr[k];
    else dxxp = pp * p.ap3spkr[k] + pc * p.ac3spkr[k] + pm * p.am3spkr[k];
    return (p.ga * h + p.ro * ru + (p.al * p.pf_d) * dxxp) * p.dt;
}

// per-routine kernels (point layout of afid_kernels.hpp)
__global__ void __launch_bounds__(256) k_explicit_phase(KP p) {
    AFID_POINT_PROLOGUE(p.nxmr, p.nyr, p.nzr)
    const double *f = p.phi;
    p.hphi[ridx(p, k, j, i)] = ex_phase_val<double>(p, f[ridx(p, k, j, i)], f[ridx(p, k, jm, i)], f[ridx(p, k, jp, i)],
                                            f[ridx(p, k, j, im)], f[ridx(p, k, j, ip)], p.tempr[ridx(p, k, j, i)]);
}
__global__ void __launch_bounds__(256) k_rhs_phase(KP p) {
    AFID_POINT_PROLOGUE(p.nxmr, p.nyr, p.nzr)
    const long long c = ridx(p, k, j, i);
    const double *f = p.phi;
    const double pm = k > 0 ? f[c - 1] : 0.0, pp = k < p.nxmr - 1 ? f[c + 1] : 0.0;
    const double h = p.hphi[c];
    p.rhsr[c] = rhs_phase_val(p, k, h, p.ruphi[c], pm, f[c], pp);
    p.ruphi[c] = h;
}
// AddVolumePenalty, phasefield.F90:525-566
__global__ void __launch_bounds__(256) k_volume_penalty(KP p) {
    AFID_POINT_PROLOGUE(p.nxm, p.ny, p.nz)
    const long long c = bidx(p, k, j, i);
    const double *pc = p.phic;
    if (k >= 1) p.qcap[c] -= (pc[c] + pc[c - 1]) * p.vx[c] * p.heta;
    p.dph[c] -= (pc[c] + pc[bidx(p, k, jm, i)]) * p.vy[c] * p.heta;
    p.dq[c] -= (pc[c] + pc[bidx(p, k, j, im)]) * p.vz[c] * p.heta;
}

// SolveImpEqnUpdate_X_pf / _YZ_pf (phasefield.F90:821-930) for the
// per-routine path: one column per wavefront, rhs as assembled by
// ImplicitAndUpdateV*, q updated in place (rows 2..nxm of vx, 1..nxm of
// vy / vz).  AX 0: vx (rows 1 and nx are identity rows with rhs -vx, rows
// kc test 0.5 (phic(kc) + phic(kc+1))); AX 1 / 2: vy / vz (phic averaged
// with the -y / -z neighbour).
template <int CH, int AX>
__global__ void __launch_bounds__(256) k_tri_update_pf(KP p, TriFactors f, const double *rhs, double *q) {
    const long long col = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (col >= (long long)p.ny * p.nz) return;
    const int lane = threadIdx.x & 63;
    const int j = int(col % p.ny), i = int(col / p.ny);
    const long long base = (long long)i * p.plane + (long long)j * p.ldx;
    const long long nbr = AX == 1 ? (long long)i * p.plane + (long long)wrapm(j, p.ny) * p.ldx
                        : AX == 2 ? (long long)wrapm(i, p.nz) * p.plane + (long long)j * p.ldx : base;
    const int n = f.n, nxm = p.nxm;
    double v[CH], a[CH], c[CH];
#pragma unroll
    for (int m = 0; m < CH; ++m) {
        const int r = lane * CH + m;
        v[m] = 0.0; a[m] = 0.0; c[m] = 0.0;
        if (r >= n) continue;
        bool solid;
        if (AX == 0) solid = (r == 0 || r == nxm) ? true : 0.5 * (p.phic[base + r] + p.phic[base + r + 1]) > 0.9;
        else solid = 0.5 * (p.phic[base + r] + p.phic[nbr + r]) > 0.9;
        if (solid) { v[m] = -q[base + r]; }
        else { v[m] = rhs[base + r] * f.s[r]; a[m] = f.a[r]; c[m] = f.c[r]; }
    }
    wave_tri_solve_general<CH>(v, a, c);
#pragma unroll
    for (int m = 0; m < CH; ++m) {
        const int r = lane * CH + m;
        if (AX == 0 ? (r >= 1 && r < nxm) : (r < n)) q[base + r] += v[m];
    }
}

// set_ice_sphere (phasefield.F90:311-341) with the radius r0 of the
// seeded initial state: refined phi = (1 - tanh((r - r0)/(2 eps)))/2 ...
template <typename RT>
__global__ void __launch_bounds__(256) k_init_phi_sphere(KP p, const double *xmr, double r0, double eps, double alx3,
                                                          double ylen, double zlen) {
    const int k = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y, i = blockIdx.z;
    if (k >= p.nxr || j >= p.nyr) return;
    const long long o = ridx(p, k, j, i);
    RT *phi = sel<RT>(p.phi, p.phif);
    if (k >= p.nxmr) { phi[o] = RT(0); return; }
    const double y = (j + 0.5) * ylen / p.nyr, z = (i + 0.5) * zlen / p.nzr;
    const double dx = xmr[k] - 0.5 * alx3, dy = y - 0.5 * ylen, dz = z - 0.5 * zlen;
    const double r = sqrt(dx * dx + dy * dy + dz * dz);
    phi[o] = RT(0.5 * (1.0 - tanh(0.5 * (r - r0) / eps)));
}
// ... and T = 0 in the base cells inside the sphere
__global__ void __launch_bounds__(256) k_init_temp_sphere(KP p, const double *xm, double r0, double alx3, double ylen,
                                                           double zlen) {
    const int k = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y, i = blockIdx.z;
    if (k >= p.nxm || j >= p.ny) return;
    const double y = (j + 0.5) * ylen / p.ny, z = (i + 0.5) * zlen / p.nz;
    const double dx = xm[k] - 0.5 * alx3, dy = y - 0.5 * ylen, dz = z - 0.5 * zlen;
    if (sqrt(dx * dx + dy * dy + dz * dz) <= r0) p.temp[bidx(p, k, j, i)] = 0.0;
}

}  // namespace afid
