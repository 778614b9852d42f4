// ibm.hpp -- immersed-boundary moving walls: marker forcing, spreading, marker motion
// and the forcing of the populations (k_Gwall, k_Gibm, k_Force of
// D3Q19_opencl/kernel.cl:3648-3807 and D3Q27_opencl/kernel.cl:2828-2986, with the helpers
// Urot/Xrot/icBox of K19:1112-1279).
//
// Markers are points in lattice coordinates (xyz interleaved, as movingSTLcList).  After
// each step:
//   gwall:  G_m = U_wall(x_m) - sum_box u(x_b) delta(x_b - x_m)   (one work-item per marker)
//   spread: G(x_b) += G_m delta(x_b - x_m) over the 8-cell box, with hardware float atomics,
//           and each touched cell enters a compact list once per step (stamp per cell);
//           then the marker moves by the translation and turns by rotOmega about the axis
//           (a marker spreads nothing but its own forcing: one kernel does both)
//   force:  f_q += rho w_q 3 (G . c_q) on the listed fluid cells only -- the reference
//           visits every cell, but G is zero away from the boxes, so the result is the same.
// The spread sums every contribution.  The reference writes the value atom_add_float
// returns (the value before the add) back into the cell (K19:3760-3762), which undoes the
// add unless another work-item interleaves: that result depends on scheduling and is not
// reproduced.  Urot/Xrot keep the reference's axis dot product OX_x*e0_z (K19:1213, 1256).
#pragma once

#include "d3q27_step.hpp"

namespace lbffs {

template <typename Real>
struct IbmMotion {
    Real trans[3];   // uMovingTrans, vMovingTrans, wMovingTrans (lattice units per step)
    Real centre[3];  // rotX, rotY, rotZ
    Real axis[3];    // rotAxisX, rotAxisY, rotAxisZ
    Real omega;      // rotOmega (radians per step)
};

// the frame of the rotation at a point (K19:1211-1233): the point's offset from the axis
// foot OOp, the radial unit vector e1, the tangential e2 = e0 x e1, and the radius
template <typename Real>
struct RotFrame {
    Real OOp[3], e1[3], e2[3], r;
};

template <typename Real>
__device__ inline RotFrame<Real> rot_frame(const IbmMotion<Real> &m, Real x, Real y, Real z)
{
    RotFrame<Real> F;
    const Real OX[3] = {x - m.centre[0], y - m.centre[1], z - m.centre[2]};
    const Real *e0 = m.axis;
    const Real OXdotE0 = OX[0] * e0[0] + OX[1] * e0[1] + OX[0] * e0[2];  // sic (K19:1213)
    Real OpX[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        F.OOp[a] = OXdotE0 * e0[a];
        OpX[a] = OX[a] - F.OOp[a];
    }
    const Real mag = sqrt(OpX[0] * OpX[0] + OpX[1] * OpX[1] + OpX[2] * OpX[2]);
#pragma unroll
    for (int a = 0; a < 3; a++) F.e1[a] = OpX[a] / mag;
    F.e2[0] = e0[1] * F.e1[2] - e0[2] * F.e1[1];
    F.e2[1] = e0[2] * F.e1[0] - e0[0] * F.e1[2];
    F.e2[2] = e0[0] * F.e1[1] - e0[1] * F.e1[0];
    F.r = sqrt(OpX[0] * OpX[0] + OpX[1] * OpX[1] + OpX[2] * OpX[2]);
    return F;
}

// trilinear weight of box corner b (0..7: +x, +y, +z bits as icBox, K19:1112-1155) of the
// cell (i, j, k) below the marker; false when the corner lies outside (no wrap)
template <typename Real>
__device__ inline bool box_corner(int b, int i, int j, int k, int nx, int ny, int nz, Real x, Real y, Real z,
                                  uint32_t &ic, Real &d)
{
    const int di = (b == 1 || b == 4 || b == 5 || b == 7) ? 1 : 0;
    const int dj = (b == 2 || b == 4 || b == 6 || b == 7) ? 1 : 0;
    const int dk = (b == 3 || b == 5 || b == 6 || b == 7) ? 1 : 0;
    const int bi = i + di, bj = j + dj, bk = k + dk;
    d = (Real(1) - fabs(Real(bi) - x)) * (Real(1) - fabs(Real(bj) - y)) * (Real(1) - fabs(Real(bk) - z));
    ic = (uint32_t)bi + (uint32_t)nx * ((uint32_t)bj + (uint32_t)ny * (uint32_t)bk);
    return bi < nx && bj < ny && bk < nz;
}

// lanes below this one whose bit is set
__device__ inline uint32_t lanes_below(uint64_t mask)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// k_Gwall (K19:3648-3716) and k_Gibm (K19:3718-3779) with a summing spread; cells touched this
// step are listed once.  What bounds it is latency and the adds to memory: markers lie closer
// than a cell, so that 64 of them in a row share their 512 corners several times over.  Where the box
// of a wave's corners has no more cells than that (markers listed along a surface), the wave sums
// them by cell in LDS and every cell touched takes one stamp and three adds to memory; otherwise
// each corner goes there itself.  The 24 velocities of a marker are
// loaded together (a corner outside the lattice reads corner 0, weightless), and a wave takes its
// list slots with one add to the counter.  One corner at a time,
// with a returning atomic and an add to the counter each, in two kernels, 6400 markers of a ring
// took 30 us per step; with their adds batched 19, with the box 8 (192x96x64 FP32 step with markers
// 63.0 -> 52.4 us).  Markers in no order (6400 over 96x64x64: 50 us either way) keep the direct adds.
constexpr int kIbmBlock = 64;
constexpr int kIbmBox = 8 * kIbmBlock;  // cells of the largest box summed in LDS
// least value over the wave's lanes (a full wave)
__device__ inline int wave_min(int v)
{
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v = min(v, __shfl_xor(v, d));
    return v;
}

template <typename Real>
__global__ void __launch_bounds__(kIbmBlock)
    ibm_spread_move_kernel(int n, Real *xyz, int nx, int ny, int nz, const Real *u, const Real *v, const Real *w,
                           IbmMotion<Real> m, Real *Gm, Real *Gx, Real *Gy, Real *Gz, uint32_t *mark, uint32_t stamp,
                           int *list, int *count, int cap)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    const bool active = p < n;
    __shared__ Real G[3][kIbmBox];
    __shared__ uint32_t touched[kIbmBox];
    Real x = 0, y = 0, z = 0, gx = 0, gy = 0, gz = 0, d[8];
    uint32_t ib[8], in = 0;  // corners; those inside the lattice
    int i = 0, j = 0, k = 0;
    if (active) {
        x = xyz[3 * p];
        y = xyz[3 * p + 1];
        z = xyz[3 * p + 2];
        i = (int)x, j = (int)y, k = (int)z;  // truncation (K19:3671-3673)
        if (i >= 0 && i < nx && j >= 0 && j < ny && k >= 0 && k < nz) {
#pragma unroll
            for (int b = 0; b < 8; b++) in |= box_corner(b, i, j, k, nx, ny, nz, x, y, z, ib[b], d[b]) ? 1u << b : 0u;
        }
        Real ui = 0, vi = 0, wi = 0;
        if (in) {
            Real cu[8], cv[8], cw[8];
#pragma unroll
            for (int b = 0; b < 8; b++) {
                const uint32_t c = (in >> b) & 1u ? ib[b] : ib[0];  // corner 0 is the cell itself
                cu[b] = u[c];
                cv[b] = v[c];
                cw[b] = w[c];
            }
#pragma unroll
            for (int b = 0; b < 8; b++) {
                const bool ok = (in >> b) & 1u;
                ui = pick(ok, ui + cu[b] * d[b], ui);
                vi = pick(ok, vi + cv[b] * d[b], vi);
                wi = pick(ok, wi + cw[b] * d[b], wi);
            }
        }
        const RotFrame<Real> F = rot_frame(m, x, y, z);
        Real U[3];
#pragma unroll
        for (int a = 0; a < 3; a++) U[a] = m.trans[a] + F.r * m.omega * F.e2[a];
        gx = U[0] - ui, gy = U[1] - vi, gz = U[2] - wi;
        Gm[p] = gx;
        Gm[n + p] = gy;
        Gm[2 * n + p] = gz;
    }
    // the box of the wave's corners (a marker outside the lattice takes no part)
    const int lox = wave_min(in ? i : nx), loy = wave_min(in ? j : ny), loz = wave_min(in ? k : nz);
    const int bx = 2 - lox - wave_min(in ? -i : 0), by = 2 - loy - wave_min(in ? -j : 0), bz = 2 - loz - wave_min(in ? -k : 0);
    const bool any = __ballot(in != 0) != 0;
    uint32_t ic[8], old[8];
#pragma unroll
    for (int b = 0; b < 8; b++) old[b] = stamp;
    if (any && (long)bx * by * bz <= kIbmBox) {
        const uint32_t cells = (uint32_t)(bx * by * bz);
        for (uint32_t e = threadIdx.x; e < cells; e += kIbmBlock) {
            touched[e] = 0;
            G[0][e] = G[1][e] = G[2][e] = Real(0);
        }
        __syncthreads();
#pragma unroll
        for (int b = 0; b < 8; b++) {
            if (!((in >> b) & 1u)) continue;
            const int di = (b == 1 || b == 4 || b == 5 || b == 7) ? 1 : 0;
            const int dj = (b == 2 || b == 4 || b == 6 || b == 7) ? 1 : 0;
            const int dk = (b == 3 || b == 5 || b == 6 || b == 7) ? 1 : 0;
            const int e = (i + di - lox) + bx * ((j + dj - loy) + by * (k + dk - loz));
            touched[e] = 1;
            atomicAdd(&G[0][e], gx * d[b]);
            atomicAdd(&G[1][e], gy * d[b]);
            atomicAdd(&G[2][e], gz * d[b]);
        }
        __syncthreads();
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const uint32_t e = (uint32_t)b * kIbmBlock + threadIdx.x;
            if (e >= cells || !touched[e]) continue;
            const uint32_t t = e / (uint32_t)bx, di = e - t * (uint32_t)bx, dk = t / (uint32_t)by, dj = t - dk * (uint32_t)by;
            ic[b] = (lox + di) + (uint32_t)nx * ((loy + dj) + (uint32_t)ny * (loz + dk));
            old[b] = atomicExch(&mark[ic[b]], stamp);
            atomicAdd(&Gx[ic[b]], G[0][e]);
            atomicAdd(&Gy[ic[b]], G[1][e]);
            atomicAdd(&Gz[ic[b]], G[2][e]);
        }
    } else {
#pragma unroll
        for (int b = 0; b < 8; b++) {
            ic[b] = ib[b];
            if ((in >> b) & 1u) old[b] = atomicExch(&mark[ib[b]], stamp);
        }
#pragma unroll
        for (int b = 0; b < 8; b++)
            if ((in >> b) & 1u) {
                atomicAdd(&Gx[ib[b]], gx * d[b]);
                atomicAdd(&Gy[ib[b]], gy * d[b]);
                atomicAdd(&Gz[ib[b]], gz * d[b]);
            }
    }
    // list slots: one add to the counter per wave, group by group in lane order after it
    uint32_t total = 0;
#pragma unroll
    for (int b = 0; b < 8; b++) total += (uint32_t)__popcll(__ballot(old[b] != stamp));
    int base = 0;
    if (total && threadIdx.x == 0) base = atomicAdd(count, (int)total);
    base = __builtin_amdgcn_readfirstlane(base);
#pragma unroll
    for (int b = 0; b < 8; b++) {
        const uint64_t mask = __ballot(old[b] != stamp);
        if (old[b] != stamp) {
            const int slot = base + (int)lanes_below(mask);
            if (slot < cap) list[slot] = (int)ic[b];
        }
        base += __popcll(mask);
    }
    if (!active) return;
    // translation, then the turn by rotOmega (Xrot, K19:1238-1279)
    const Real xt = x + m.trans[0], yt = y + m.trans[1], zt = z + m.trans[2];
    const RotFrame<Real> F = rot_frame(m, xt, yt, zt);
    const Real c = cos(m.omega), s = sin(m.omega);
    xyz[3 * p] = m.centre[0] + F.OOp[0] + F.r * (c * F.e1[0] + s * F.e2[0]);
    xyz[3 * p + 1] = m.centre[1] + F.OOp[1] + F.r * (c * F.e1[1] + s * F.e2[1]);
    xyz[3 * p + 2] = m.centre[2] + F.OOp[2] + F.r * (c * F.e1[2] + s * F.e2[2]);
}

// k_Force (K19:3781-3807) on the listed cells; zero_after clears G behind it so that the
// next step spreads into zeros.  Thread 0 clears the counter of the next step's list.  All
// populations are loaded before the first is stored: stored one by one, each load waited for
// the store before it (18.6 us per step for 6400 markers, now 8.4).
template <typename S, typename Real, int Q>
__global__ void __launch_bounds__(kIbmBlock)
    ibm_force_kernel(const int *list, const int *count, int *next_count, int cap, size_t fs, S *f,
                     const uint16_t *flag, const Real *rho, Real *Gx, Real *Gy, Real *Gz, int zero_after)
{
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx == 0) *next_count = 0;
    const int cnt = min(*count, cap);
    if (idx >= cnt) return;
    const uint32_t ic = (uint32_t)list[idx];
    const Real gx = Gx[ic], gy = Gy[ic], gz = Gz[ic];
    if (zero_after) {
        Gx[ic] = Real(0);
        Gy[ic] = Real(0);
        Gz[ic] = Real(0);
    }
    if (flag[ic] & F_SOLID) return;
    const Real r3 = rho[ic] * Real(3);
    S raw[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) raw[q] = f[pop_at<Q, S>(q, ic, fs)];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int cx = Q == 27 ? L27::cx[q] : L19::cx[q];
        const int cy = Q == 27 ? L27::cy[q] : L19::cy[q];
        const int cz = Q == 27 ? L27::cz[q] : L19::cz[q];
        const Real wqq = wq<Real, Q>(q);
        const Real fq = Codec<S, Real, Q>::load(&raw[q], q, wqq);
        Codec<S, Real, Q>::store(f + pop_at<Q, S>(q, ic, fs), fq + r3 * wqq * (gx * Real(cx) + gy * Real(cy) + gz * Real(cz)),
                                 q, wqq);
    }
}

// G of the cells listed by the last spread back to zero (start of a call after a call
// whose last step kept them for output)
template <typename Real>
__global__ void ibm_zero_listed_kernel(const int *list, const int *count, int cap, Real *Gx, Real *Gy, Real *Gz)
{
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= min(*count, cap)) return;
    const int ic = list[idx];
    Gx[ic] = Real(0);
    Gy[ic] = Real(0);
    Gz[ic] = Real(0);
}

template <typename Real>
__global__ void fill_kernel(Real *p, size_t n, Real v)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

}  // namespace lbffs
