// d3q19_step.hpp -- the fused D3Q19 time-step kernel.
//
// One work-item per cell, cells flattened as ic = i + nx*(j + ny*k) so that a
// wavefront's 64 lanes touch 64 consecutive cells of one direction (in a population block
// or a direction array, pop_at): every store is a coalesced run of 256 B (FP32) or 128 B
// (16-bit), every pull one or two.
// The kernel does, for each fluid cell, what k_streamingCollision does
// (D3Q19_opencl/kernel.cl:3547-3645):
//   pull streaming (interior: fixed offsets; faces: wrap or wall per face code),
//   fixed-velocity / fixed-density / wall-function / outlet face conditions,
//   simple bounce-back on solid links with momentum-exchange force,
//   moments, sub-grid model (WALE or Smagorinsky), sponge, recursive-regularized
//   collision with the dpdx body force.
// Deliberate differences from the reference's data flow (results are unchanged):
//   * neighbour reads of rho/u/v/w see the previous step (Jacobi) instead of a
//     scheduling-dependent mix, via two macro buffers that alternate each step;
//   * 19 per-cell side arrays are replaced by one 16-bit flag word; side arrays are
//     read only by the cells whose flag asks for them;
//   * rho/u/v/w/tauSGS/Fw/G are written for every cell only when the caller asks
//     (last step of a call or store_every), otherwise only where later steps read them.
#pragma once

#include "lbffs_common.hpp"

namespace lbffs {

// D3Q19 directions (kernel.cl:3558-3560) as compile-time tables, so that unrolled
// loops fold the lattice constants into the instruction stream
struct L19 {
    static constexpr int cx[19] = {0, 1, -1, 0, 0, 0, 0, 1, -1, 1, -1, 1, -1, 1, -1, 0, 0, 0, 0};
    static constexpr int cy[19] = {0, 0, 0, 1, -1, 0, 0, 1, -1, -1, 1, 0, 0, 0, 0, 1, -1, 1, -1};
    static constexpr int cz[19] = {0, 0, 0, 0, 0, 1, -1, 0, 0, 0, 0, 1, -1, -1, 1, 1, -1, -1, 1};
    __host__ __device__ static constexpr int opp(int q) { return q == 0 ? 0 : ((q & 1) ? q + 1 : q - 1); }
    // diagonals with the x, y or z component flipped; the other directions reversed
    static constexpr int mirx[19] = {0, 2, 1, 4, 3, 6, 5, 10, 9, 8, 7, 14, 13, 12, 11, 16, 15, 18, 17};
    static constexpr int miry[19] = {0, 2, 1, 4, 3, 6, 5, 9, 10, 7, 8, 12, 11, 14, 13, 18, 17, 16, 15};
    static constexpr int mirz[19] = {0, 2, 1, 4, 3, 6, 5, 8, 7, 10, 9, 13, 14, 11, 12, 17, 18, 15, 16};
};

template <typename Real>
__host__ __device__ constexpr Real w19(int q)
{
    return q == 0 ? Real(1) / Real(3) : (q <= 6 ? Real(1) / Real(18) : Real(1) / Real(36));
}

// Arguments of one step launch, shared by the D3Q19 and D3Q27 kernels.
template <typename Real, int Q>
struct StepArgs {
    uint32_t N;
    uint32_t fstride;  // 16-bit values: elements between two direction arrays (pop_at)
    int keep;          // 1: the new populations stay in the caches (fits_cache)
    int wave_runs;     // 1: a wave of the cell order holds one aligned run of 64 cells
    int nx, ny, nz;
    FastDiv dnx, dny;
    int off[Q];  // interior pull offset: source = ic - off[q]
    const void *fsrc;
    void *fdst;
    const uint16_t *flag;
    const Real *u0, *v0, *w0, *sdf, *omega;
    const Real *rho_o, *u_o, *v_o, *w_o;  // macros of the previous step
    Real *rho_n, *u_n, *v_n, *w_n;        // macros written by this step
    Real *tau, *Fwx, *Fwy, *Fwz, *Gx, *Gy, *Gz;
    Real dpdx, LES, omegaB, spz, Cs, omega0;
    Real clim;  // cumulant limiter (D3Q27)
    const Real *qlink;  // q-distances of the solid links (Q*N, q-major), read when ibb
    int ibb;            // interpolated bounce-back with qlink instead of the reference's walls
    int sround;         // 16-bit forms: stochastic rounding of the stored deviations
    int damping;
    int mac_all;      // write u/v/w for every fluid cell
    int rho_all;      // write rho for every fluid cell (implies mac_all)
    int aux_all;      // write tauSGS / Fw / G for every fluid cell
    int sponge_mask;  // faces whose centre cell is Outlet or FixedDensity (tauSpongeZone)
    Real inv_spx, inv_spy, inv_spz;  // 1 / (n * spzWidth) per axis
    int tune;         // TUNE_* launch options chosen by the autotuner
    // y-tiled cell order (TUNE_YTILE): tiles of ty rows, plane by plane inside a tile
    uint32_t tile_cells, tile_plane, nxny;  // nx*ty*nz, nx*ty, nx*ny
    FastDiv dtile, dplane;
    const uint32_t *fcells;  // the lattice's non-solid face cells (the face pass runs these)
    uint32_t nface;
    const uint32_t *wclass;  // per-wave summary (wave_class), or null: every wave reads its flags first
    int coll;                 // D3Q27: LBFFS_COLL_RR or LBFFS_COLL_CUMULANT (uniform per launch)
    uint32_t step;            // step number (stochastic rounding), see sr_step
    const uint32_t *step_ctr; // batches: device counter of the steps run in the current call
};

template <typename Real>
using Step19Args = StepArgs<Real, 19>;

// launch options (uniform per launch)
enum : int {
    TUNE_NT_STORE = 1,  // the populations are stored non-temporally whatever the lattice's size (keep)
    TUNE_NO_XCD = 2,    // keep the hardware work-group order (no XCD slab remap)
    TUNE_YTILE = 4,     // visit the cells in y-tiles (see ytile_cell)
    TUNE_SPLIT = 8,     // two passes per step: the cells off the faces, then the face cells
    TUNE_NO_PURE = 16,  // every wave waits for its flags before it pulls (no per-wave summary)
    TUNE_FACE_FIRST = 32,  // one launch: the face-list work-groups first, then the cells off the faces
    TUNE_XCD_CHUNK = 64,   // deal runs of kXcdChunk consecutive blocks to each XCD in turn
};

// the face pass skips the face cells that the interior pass updates in their own waves:
// those of XMIX and WRAP waves.  (Handing the x-face cells of XMIX waves to the face pass
// instead is slower on every lattice measured: consecutive x-face cells of the list lie a
// row apart, so each lane's pulls touch cache lines of their own, where in their own wave
// they share the lines of their neighbours' pulls.)
__device__ inline bool face_pass_skips(uint32_t cls)
{
    return cls == WAVE_WRAP || cls == WAVE_XMIX;
}

// Cell of position lin in the y-tiled order: tiles of ty full rows (ny a multiple of ty),
// each walked plane by plane (k), row by row inside a plane.  The velocity gradient of
// WALE reads the planes k - 1 and k + 1 of a cell's velocities: over a tile of 32 rows of
// 1024 cells those three planes of three arrays take 1.2 MB and stay in one XCD's L2
// between their uses, where whole planes (1.5 MB each) do not.
template <typename A>
__device__ inline uint32_t ytile_cell(const A &a, uint32_t lin)
{
    const uint32_t tile = fdiv(lin, a.dtile);
    const uint32_t rem = lin - tile * a.tile_cells;
    const uint32_t k = fdiv(rem, a.dplane);
    return (rem - k * a.tile_plane) + tile * a.tile_plane + k * a.nxny;
}

// XCD-aware block order: the hardware deals work-groups round-robin over the 8 XCDs;
// renumber them so that each XCD walks one contiguous slab of cells and the partial
// cache lines at block edges are shared inside one L2.
__device__ inline uint32_t xcd_block(uint32_t pid, uint32_t G)
{
    const uint32_t nx = 8;
    uint32_t x = pid % nx, local = pid / nx;
    uint32_t base = G / nx, r = G % nx;
    return x * base + (x < r ? x : r) + local;
}

// XCD-chunked block order: the k-th work-group of XCD x (hardware block 8k + x) takes block
// (k / C) 8C + x C + k mod C, so each XCD runs C consecutive blocks while the eight XCDs
// still sweep one contiguous front of the arrays.  A pull shifted by one cell in x reads
// one cache line of its neighbour block; in hardware order that neighbour runs on another
// XCD and the line is fetched twice (once per L2), in chunks only every C-th block edge
// crosses XCDs.  The blocks past the last whole group of 8C keep their own number.
// Eight blocks (2048 cells: the rows beside a row of a few hundred cells run on the same XCD,
// which the velocity gradient reads) measured as fast as or faster than 4, 16 and 64:
// backstep 768x192x128 FP32 466 us per step (4: 474, 16: 464, 64: 470; hardware order 472,
// slabs 483), D3Q19 WALE channel 160x128x128 85.8 us (87.5, 85.9, 87.1; 88.4, 90.1).
constexpr uint32_t kXcdChunk = 8;
__device__ inline uint32_t xcd_chunk_block(uint32_t g, uint32_t G)
{
    constexpr uint32_t span = 8 * kXcdChunk;
    if (g >= G - G % span) return g;
    const uint32_t k = g / 8, x = g % 8;
    return (k / kXcdChunk) * span + x * kXcdChunk + k % kXcdChunk;
}

// block g of G in the order the launch option asks for; g % 8 must be the XCD that the
// hardware gives block g (true when the blocks before the first are a multiple of 8)
__device__ inline uint32_t ordered_block(uint32_t g, uint32_t G, uint32_t tune)
{
    if (tune & TUNE_XCD_CHUNK) return xcd_chunk_block(g, G);
    return (tune & TUNE_NO_XCD) ? g : xcd_block(g, G);
}

// pull source for a face cell (kernel.cl:328-575 upwindID_B): wrap across non-wall faces,
// -1 for a link through a wall face.
// Formed from the interior source ic - c_q in 32-bit arithmetic: a crossed periodic face moves
// the source by a whole row (x), plane (y) or lattice (z), c_x nx, c_y nx ny or c_z nx ny nz
// cells; unsigned wrap-around is exact because the result lies in the lattice.
__device__ inline long face_upwind(int q, long ic, int i, int j, int k, int nx, int ny, int nz, int b1, int b2, int b3)
{
    const int cx = L19::cx[q], cy = L19::cy[q], cz = L19::cz[q];
    const bool crx = cx == 1 ? i == 0 : (cx == -1 ? i == nx - 1 : false);
    const bool cry = cy == 1 ? j == 0 : (cy == -1 ? j == ny - 1 : false);
    const bool crz = cz == 1 ? k == 0 : (cz == -1 ? k == nz - 1 : false);
    if ((crx && is_wall_code(b1)) || (cry && is_wall_code(b2)) || (crz && is_wall_code(b3))) return -1;
    const uint32_t nxny = (uint32_t)nx * (uint32_t)ny;
    uint32_t s = (uint32_t)ic - (uint32_t)cx - (uint32_t)cy * (uint32_t)nx - (uint32_t)cz * nxny;
    if (crx) s += (uint32_t)cx * (uint32_t)nx;
    if (cry) s += (uint32_t)cy * nxny;
    if (crz) s += (uint32_t)cz * nxny * (uint32_t)nz;
    return (long)s;
}

// kernel.cl:105-326 reflectOrMirrorQ as table lookups: the bounce-back partner, with
// Symmetry faces flipping only the normal component of diagonal directions -- of the first
// of its axes, in the order x, y, z, whose code is Symmetry.  (Selects between constants once
// q is: a face cell's pull takes its reflected slot from here.)
__device__ inline int mirror_q(int q, int b1, int b2, int b3)
{
    int r = L19::opp(q);
    if (q <= 6) return r;
    if (L19::cz[q] != 0) r = (b3 == BC_SYMMETRY) ? L19::mirz[q] : r;
    if (L19::cy[q] != 0) r = (b2 == BC_SYMMETRY) ? L19::miry[q] : r;
    if (L19::cx[q] != 0) r = (b1 == BC_SYMMETRY) ? L19::mirx[q] : r;
    return r;
}

// kernel.cl:1346-1395 cornerFlag
__device__ inline int corner_flag(int b3, int i, int j, int k, int nx, int ny, int nz)
{
    bool xi = (i == 0 || i == nx - 1), yj = (j == 0 || j == ny - 1), zk = (k == 0 || k == nz - 1);
    if (nz - 1 == 0 || b3 == 0) return (xi && yj) ? 1 : 0;
    return ((xi && yj) || (xi && zk) || (yj && zk)) ? 1 : 0;
}

// kernel.cl:1621-1652 calcTauw (Newton on the wall law; the loop's error test uses
// the initial y+ as the reference does, K19:1646)
template <typename Real>
__device__ inline Real calc_tauw(Real rhow, Real magUp, Real nu)
{
    const Real y = Real(1.5), kappa = Real(0.42), E = Real(9.1);
    Real ut = sqrt(nu * magUp);
    int iter = 0;
    Real err;
    const Real yPlus = y * ut / nu;
    do {
        Real kUu = fmin(kappa * magUp / ut, Real(50));
        Real fkUu = exp(kUu) - Real(1) - kUu * (Real(1) + Real(0.5) * kUu);
        Real func = -ut * y / nu + magUp / ut + (fkUu - kUu * kUu * kUu / Real(6)) / E;
        Real dfunc = y / nu + magUp / (ut * ut) + (kUu * fkUu / ut) / E;
        ut = ut + func / dfunc;
        err = fabs(yPlus - y * ut / nu);
    } while (err > Real(0.005) && ++iter < 100);
    ut = fmax(ut, Real(0));
    return rhow * ut * ut;
}

// sum of the populations that leave through a face plus twice those arriving (Zou-He
// wall density numerator); dir 0/1/2 = x/y/z, lo = min face
template <typename Real>
__device__ inline Real zouhe_sum(const Real *ft, int dir, bool lo)
{
    Real s = Real(0), t = Real(0);
    // tangential populations in the reference's summation order
    if (dir == 0) {
        s = ft[0] + ft[3] + ft[4] + ft[5] + ft[6] + ft[15] + ft[16] + ft[17] + ft[18];
        t = lo ? (ft[2] + ft[10] + ft[8] + ft[14] + ft[12]) : (ft[1] + ft[7] + ft[9] + ft[11] + ft[13]);
    } else if (dir == 1) {
        s = ft[0] + ft[1] + ft[2] + ft[5] + ft[6] + ft[11] + ft[12] + ft[14] + ft[13];
        t = lo ? (ft[4] + ft[9] + ft[8] + ft[18] + ft[16]) : (ft[3] + ft[7] + ft[10] + ft[15] + ft[17]);
    } else {
        s = ft[0] + ft[1] + ft[2] + ft[3] + ft[4] + ft[7] + ft[8] + ft[9] + ft[10];
        t = lo ? (ft[6] + ft[12] + ft[13] + ft[16] + ft[17]) : (ft[5] + ft[14] + ft[11] + ft[18] + ft[15]);
    }
    return s + Real(2) * t;
}

// c ? a : b of two values (a conditional on ft[] elements themselves would name one of two
// addresses, and put ft[] in memory)
template <typename T>
__device__ inline T pick(bool c, T a, T b)
{
    return c ? a : b;
}

// Ladd moving-wall correction of the five populations entering through a face with
// wall velocity (un, ut1, ut2) = (normal, first tangential, second tangential),
// kernel.cl:1397-1512.  Written with value selects (never "if (lo) ft[a] else ft[b]")
// so that ft[] stays in registers.
template <int A0, int A1, int A2, int A3, int A4, int B0, int B1, int B2, int B3, int B4, typename Real>
__device__ inline void ladd_face(Real *ft, bool lo, Real rhow, Real un, Real ut1, Real ut2)
{
    const Real d0 = rhow * un / Real(3);
    const Real d1 = rhow * (un + ut1) / Real(6);
    const Real d2 = rhow * (un - ut1) / Real(6);
    const Real d3 = rhow * (un + ut2) / Real(6);
    const Real d4 = rhow * (un - ut2) / Real(6);
    ft[A0] = lo ? ft[A0] + d0 : ft[A0];
    ft[A1] = lo ? ft[A1] + d1 : ft[A1];
    ft[A2] = lo ? ft[A2] + d2 : ft[A2];
    ft[A3] = lo ? ft[A3] + d3 : ft[A3];
    ft[A4] = lo ? ft[A4] + d4 : ft[A4];
    ft[B0] = lo ? ft[B0] : ft[B0] - d0;
    ft[B1] = lo ? ft[B1] : ft[B1] - d1;
    ft[B2] = lo ? ft[B2] : ft[B2] - d2;
    ft[B3] = lo ? ft[B3] : ft[B3] - d3;
    ft[B4] = lo ? ft[B4] : ft[B4] - d4;
}

template <typename Real>
__device__ inline void ladd(Real *ft, int dir, bool lo, Real rhow, Real un, Real ut1, Real ut2)
{
    if (dir == 0)  // tangentials v, w
        ladd_face<1, 7, 9, 11, 13, 2, 8, 10, 12, 14>(ft, lo, rhow, un, ut1, ut2);
    else if (dir == 1)  // tangentials u, w
        ladd_face<3, 7, 10, 15, 17, 4, 8, 9, 16, 18>(ft, lo, rhow, un, ut1, ut2);
    else  // tangentials u, v
        ladd_face<5, 11, 14, 15, 18, 6, 12, 13, 16, 17>(ft, lo, rhow, un, ut1, ut2);
}

template <typename Real>
struct Cell {
    long ic;
    int i, j, k;
};

// derivative of one component along an axis as kernel.cl:2275-2304 forms it: central inside;
// on a face one-sided, with the cell's own value the new one (the reference reads it back
// from the array it has just written); 0 for the z gradient at k = 0 (K19:2283, a - a) and on
// a 2-D lattice.  Both neighbours are loaded, the cell itself in place of one outside the
// lattice, and the form is chosen by selects: a branch per face and component left the nine
// derivatives of a face wave waiting for memory one after another.
template <int DIR, typename Real>
__device__ inline Real grad_comp(const Real *old, Real self, uint32_t ic, int pos, int n, uint32_t stride)
{
    const bool lo = (pos == 0), hi = (pos == n - 1);
    const Real p = old[hi ? ic : ic + stride], m = old[lo ? ic : ic - stride];
    const Real inside = Real(0.5) * (p - m);
    if (DIR == 2) return n == 1 ? Real(0) : (lo ? p - p : (hi ? self - m : inside));
    return lo ? p - self : (hi ? self - m : inside);
}

// x / 3 as the division rounds it: the product with fl(1/3) and one correction by the exact
// remainder (equal to x / 3.0f for every finite float, checked exhaustively), 3 instructions
// where the division takes 10.  FP64 divides.
__device__ inline float div3(float x)
{
    const float z = 1.0f / 3.0f;
    const float q = x * z;
    return __builtin_fmaf(__builtin_fmaf(-3.0f, q, x), z, q);
}
__device__ inline double div3(double x) { return x / 3.0; }

// square root of x in [2^-96, inf], correctly rounded as sqrt() is: the hardware's value is
// within one ulp, and the signs of the remainders x - (s -+ 1 ulp) s tell which of the three
// neighbours is nearest.  sqrt() adds the scaling of tiny arguments and the tests for 0, inf
// and NaN around the same correction, 23 instructions against 8.
__device__ inline float sqrt_normal(float x)
{
    const float s = __builtin_amdgcn_sqrtf(x);
    const float dn = __uint_as_float(__float_as_uint(s) - 1u), up = __uint_as_float(__float_as_uint(s) + 1u);
    const float rd = __builtin_fmaf(-dn, s, x), ru = __builtin_fmaf(-up, s, x);
    const float r = rd <= 0.0f ? dn : s;
    return ru > 0.0f ? up : r;
}
__device__ inline double sqrt_normal(double x) { return sqrt(x); }

// kernel.cl:2267-2365 waleTauSGS (Cw = 0.325) from the velocity gradient.  The D3Q27 step is
// bound by vector issue and the D3Q19 step near it: hence div3 and sqrt_normal (both sums
// are above 1e-24 where they are used).
template <typename Real>
__device__ inline Real wale_from_grad(Real dudx, Real dudy, Real dudz, Real dvdx, Real dvdy, Real dvdz, Real dwdx,
                                      Real dwdy, Real dwdz)
{
    const Real Cw = Real(0.325);
    Real S12 = Real(0.5) * (dudy + dvdx), S13 = Real(0.5) * (dudz + dwdx), S23 = Real(0.5) * (dvdz + dwdy);
    Real SS = dudx * dudx + Real(2) * S12 * S12 + Real(2) * S13 * S13 + dvdy * dvdy + Real(2) * S23 * S23
              + dwdz * dwdz;
    // g = grad(u)^2 (g_ab = sum_c d_c u_a ... as the reference composes it)
    Real g11 = dudx * dudx + dvdx * dudy + dwdx * dudz;
    Real g12 = dudx * dvdx + dvdx * dvdy + dwdx * dvdz;
    Real g13 = dudx * dwdx + dvdx * dwdy + dwdx * dwdz;
    Real g21 = dudy * dudx + dvdy * dudy + dwdy * dudz;
    Real g22 = dudy * dvdx + dvdy * dvdy + dwdy * dvdz;
    Real g23 = dudy * dwdx + dvdy * dwdy + dwdy * dwdz;
    Real g31 = dudz * dudx + dvdz * dudy + dwdz * dudz;
    Real g32 = dudz * dvdx + dvdz * dvdy + dwdz * dvdz;
    Real g33 = dudz * dwdx + dvdz * dwdy + dwdz * dwdz;
    Real tr3 = div3(g11 + g22 + g33);
    Real d11 = g11 - tr3, d22 = g22 - tr3, d33 = g33 - tr3;
    Real d12 = Real(0.5) * (g12 + g21), d13 = Real(0.5) * (g13 + g31), d23 = Real(0.5) * (g23 + g32);
    Real SdSd = d11 * d11 + d22 * d22 + d33 * d33 + Real(2) * (d12 * d12 + d13 * d13 + d23 * d23);
    if (!(SS > Real(1e-24) && SdSd > Real(1e-24))) return Real(0);
    const Real rSd = sqrt_normal(SdSd);
    Real sd15 = SdSd * rSd;                 // SdSd^1.5
    Real ss25 = SS * SS * sqrt_normal(SS);  // SS^2.5
    Real sd125 = SdSd * sqrt_normal(rSd);   // SdSd^1.25
    return Real(9) * (Cw * Cw * sd15 / (ss25 + sd125));
}

// central difference 0.5 (p[o + d] - p[o - d]) at byte offset o (32-bit offsets from the
// array base; d = one element for x, so that it folds into the load's immediate offset)
template <typename Real>
__device__ inline Real cdiff(const Real *p, uint32_t o, uint32_t d)
{
    const char *b = (const char *)p;
    return Real(0.5) * (*(const Real *)(b + (size_t)(o + d)) - *(const Real *)(b + (size_t)(o - d)));
}

// Interior: take the central differences of interior cells directly (every step kernel;
// in the batch kernel it costs a wave per SIMD and still gains 2 %)
template <bool Interior, typename Real, int Q>
__device__ inline Real wale_tau(const StepArgs<Real, Q> &a, long ic, int i, int j, int k, Real u, Real v, Real w)
{
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    // the choice is uniform over the wave (every active lane must allow the shorter form), so
    // that a wave with a face cell runs one form and waits once for its loads
    const bool yz_in = j > 0 && j < ny - 1 && k > 0 && k < nz - 1;
    const bool all_yz_in = Interior && nx >= 3 && __ballot(!yz_in) == 0;
    if (Q == 27 && all_yz_in && __ballot(!(i > 0 && i < nx - 1)) == 0) {
        // all six neighbours exist: central differences only, as grad_comp takes them there
        const uint32_t o = (uint32_t)ic * (uint32_t)sizeof(Real);
        const uint32_t dx = (uint32_t)sizeof(Real), dy = (uint32_t)nx * dx, dz = (uint32_t)ny * dy;
        const Real *U = a.u_o, *V = a.v_o, *W = a.w_o;
        return wale_from_grad<Real>(cdiff(U, o, dx), cdiff(U, o, dy), cdiff(U, o, dz), cdiff(V, o, dx), cdiff(V, o, dy),
                                    cdiff(V, o, dz), cdiff(W, o, dx), cdiff(W, o, dy), cdiff(W, o, dz));
    }
    if (all_yz_in) {
        // (waves with x-face cells, and on D3Q19 every wave inside in y and z) the y and z
        // neighbours exist: central differences there, as grad_comp takes them; along x
        // central differences inside and, on an x face, grad_comp's one-sided difference with
        // the cell's own new velocity -- as a per-lane choice, so that such a wave runs one
        // path.  The x neighbours read on a face (the previous row's last or the next row's
        // first cell) exist, j being interior, and are not used there.
        const uint32_t o = (uint32_t)ic * (uint32_t)sizeof(Real);
        const uint32_t dx = (uint32_t)sizeof(Real), dy = (uint32_t)nx * dx, dz = (uint32_t)ny * dy;
        const Real *U = a.u_o, *V = a.v_o, *W = a.w_o;
        const bool xlo = (i == 0), xhi = (i == nx - 1);
        auto ddx = [&](const Real *P, Real self) {
            const char *b = (const char *)P;
            const Real p = *(const Real *)(b + (size_t)(o + dx)), m = *(const Real *)(b + (size_t)(o - dx));
            return xlo ? p - self : (xhi ? self - m : Real(0.5) * (p - m));
        };
        return wale_from_grad<Real>(ddx(U, u), cdiff(U, o, dy), cdiff(U, o, dz), ddx(V, v), cdiff(V, o, dy),
                                    cdiff(V, o, dz), ddx(W, w), cdiff(W, o, dy), cdiff(W, o, dz));
    }
    const uint32_t c = (uint32_t)ic, sy = (uint32_t)nx, sz = sy * (uint32_t)ny;
    auto row = [&](const Real *P, Real self, Real &dx, Real &dy, Real &dz) {
        dx = grad_comp<0>(P, self, c, i, nx, 1u);
        dy = grad_comp<1>(P, self, c, j, ny, sy);
        dz = grad_comp<2>(P, self, c, k, nz, sz);
    };
    Real dudx, dudy, dudz, dvdx, dvdy, dvdz, dwdx, dwdy, dwdz;
    row(a.u_o, u, dudx, dudy, dudz);
    row(a.v_o, v, dvdx, dvdy, dvdz);
    row(a.w_o, w, dwdx, dwdy, dwdz);
    return wale_from_grad<Real>(dudx, dudy, dudz, dvdx, dvdy, dvdz, dwdx, dwdy, dwdz);
}

// What a cell needs beside its populations, loaded before anything is known of it (the latency
// form of the step, PASS 4 of step19_kernel): its face velocity and, for WALE, the velocities of
// its six neighbours, the cell itself in place of one outside the lattice.
template <typename Real, bool WALE>
struct EarlyLoads {
    Real u0, v0, w0;
    Real m[3][3], p[3][3];  // [component][axis]: the neighbour below and above
};
template <typename Real, bool WALE, int Q>
__device__ __forceinline__ void early_loads(EarlyLoads<Real, WALE> &e, const StepArgs<Real, Q> &a, uint32_t ic, int i, int j,
                                           int k)
{
    e.u0 = a.u0[ic];
    e.v0 = a.v0[ic];
    e.w0 = a.w0[ic];
    if constexpr (WALE) {
        const uint32_t sy = (uint32_t)a.nx, sz = sy * (uint32_t)a.ny;
        const Real *const P[3] = {a.u_o, a.v_o, a.w_o};
        const uint32_t up[3] = {i == a.nx - 1 ? ic : ic + 1u, j == a.ny - 1 ? ic : ic + sy, k == a.nz - 1 ? ic : ic + sz};
        const uint32_t dn[3] = {i == 0 ? ic : ic - 1u, j == 0 ? ic : ic - sy, k == 0 ? ic : ic - sz};
#pragma unroll
        for (int c = 0; c < 3; c++)
#pragma unroll
            for (int x = 0; x < 3; x++) {
                e.p[c][x] = P[c][up[x]];
                e.m[c][x] = P[c][dn[x]];
            }
    }
}

// wale_tau from the loaded neighbours: grad_comp's differences
template <typename Real, int Q>
__device__ __forceinline__ Real wale_tau_early(const StepArgs<Real, Q> &a, const EarlyLoads<Real, true> &e, int i, int j, int k,
                                              Real u, Real v, Real w)
{
    auto diff = [](Real p, Real m, Real self, int pos, int n) {
        return pos == 0 ? p - self : (pos == n - 1 ? self - m : Real(0.5) * (p - m));
    };
    auto diffz = [&](Real p, Real m, Real self) {
        return a.nz == 1 ? Real(0) : (k == 0 ? p - p : (k == a.nz - 1 ? self - m : Real(0.5) * (p - m)));
    };
    return wale_from_grad<Real>(
        diff(e.p[0][0], e.m[0][0], u, i, a.nx), diff(e.p[0][1], e.m[0][1], u, j, a.ny), diffz(e.p[0][2], e.m[0][2], u),
        diff(e.p[1][0], e.m[1][0], v, i, a.nx), diff(e.p[1][1], e.m[1][1], v, j, a.ny), diffz(e.p[1][2], e.m[1][2], v),
        diff(e.p[2][0], e.m[2][0], w, i, a.nx), diff(e.p[2][1], e.m[2][1], w, j, a.ny), diffz(e.p[2][2], e.m[2][2], w));
}

// reciprocal: one v_rcp_f32 in FP32 (<= 1 ulp), an exact quotient in FP64
__device__ inline float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ inline double rcp(double x) { return 1.0 / x; }
// reciprocal refined by one Newton step (e = 1 - x r, r += r e): unbiased to within
// rounding, as a division would be.  Used for 1/rho, whose error the collision turns into
// momentum (the output momentum is rho times the velocity it was given), so that a
// one-sided error of the hardware reciprocal cannot accumulate over steps.
__device__ inline float rcp_nr(float x)
{
    const float r = __builtin_amdgcn_rcpf(x);
    const float e = __builtin_fmaf(-x, r, 1.0f);
    return __builtin_fmaf(r, e, r);
}
__device__ inline double rcp_nr(double x) { return 1.0 / x; }
// square root: one v_sqrt_f32 in FP32 (<= 1 ulp), the correctly rounded one in FP64
__device__ inline float fsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ inline double fsqrt(double x) { return sqrt(x); }

// Density, momentum and the second moments sum_q c_a c_b f_q of the streamed
// populations; shared by the moments update, the Smagorinsky model and the collision.
template <typename Real>
struct Mom19 {
    Real rho, mx, my, mz;
    Real sxx, syy, szz, sxy, sxz, syz;
};

template <typename Real>
__device__ inline Mom19<Real> moments19(const Real *ft)
{
    Mom19<Real> m;
    const Real a12 = ft[1] + ft[2], a34 = ft[3] + ft[4], a56 = ft[5] + ft[6];
    const Real p78 = ft[7] + ft[8], p910 = ft[9] + ft[10], p1112 = ft[11] + ft[12], p1314 = ft[13] + ft[14];
    const Real p1516 = ft[15] + ft[16], p1718 = ft[17] + ft[18];
    m.rho = ft[0] + a12 + a34 + a56 + p78 + p910 + p1112 + p1314 + p1516 + p1718;
    const Real d78 = ft[7] - ft[8], d910 = ft[9] - ft[10], d1112 = ft[11] - ft[12], d1314 = ft[13] - ft[14];
    const Real d1516 = ft[15] - ft[16], d1718 = ft[17] - ft[18];
    m.mx = (ft[1] - ft[2]) + d78 + d910 + d1112 + d1314;
    m.my = (ft[3] - ft[4]) + d78 - d910 + d1516 + d1718;
    m.mz = (ft[5] - ft[6]) + d1112 - d1314 + d1516 - d1718;
    m.sxx = a12 + p78 + p910 + p1112 + p1314;
    m.syy = a34 + p78 + p910 + p1516 + p1718;
    m.szz = a56 + p1112 + p1314 + p1516 + p1718;
    m.sxy = p78 - p910;
    m.sxz = p1112 - p1314;
    m.syz = p1516 - p1718;
    return m;
}

// The same moments for populations held as 16-bit deviations from the weights: density
// and second moments are formed from the deviations f_q - w_q (exact differences, the
// populations being within a factor of two of their weights) plus the exact weight moments
// (sum w_q = 1, sum w_q c_a c_b = delta_ab / 3).  Summed as w_q + deviation, the density
// would carry the FP32 weights' excess sum_q fl(w_q) - 1 (about 2 ulp of 1) below every
// deviation a 16-bit value can hold, and its rounding to FP32 would go the same way in
// every cell and every step: a closed lattice would gain mass at about 1e-7 per cell per
// step, whatever the 16-bit rounding.  The momentum sums pairwise differences, as above.
template <typename Real>
__device__ inline Mom19<Real> moments19_dev(const Real *ft)
{
    Real d[19];
#pragma unroll
    for (int q = 0; q < 19; q++) d[q] = ft[q] - w19<Real>(q);
    Mom19<Real> m;
    const Real a12 = d[1] + d[2], a34 = d[3] + d[4], a56 = d[5] + d[6];
    const Real p78 = d[7] + d[8], p910 = d[9] + d[10], p1112 = d[11] + d[12], p1314 = d[13] + d[14];
    const Real p1516 = d[15] + d[16], p1718 = d[17] + d[18];
    m.rho = Real(1) + (d[0] + a12 + a34 + a56 + p78 + p910 + p1112 + p1314 + p1516 + p1718);
    const Real d78 = d[7] - d[8], d910 = d[9] - d[10], d1112 = d[11] - d[12], d1314 = d[13] - d[14];
    const Real d1516 = d[15] - d[16], d1718 = d[17] - d[18];
    m.mx = (d[1] - d[2]) + d78 + d910 + d1112 + d1314;
    m.my = (d[3] - d[4]) + d78 - d910 + d1516 + d1718;
    m.mz = (d[5] - d[6]) + d1112 - d1314 + d1516 - d1718;
    const Real third = Real(1) / Real(3);
    m.sxx = third + (a12 + p78 + p910 + p1112 + p1314);
    m.syy = third + (a34 + p78 + p910 + p1516 + p1718);
    m.szz = third + (a56 + p1112 + p1314 + p1516 + p1718);
    m.sxy = p78 - p910;
    m.sxz = p1112 - p1314;
    m.syz = p1516 - p1718;
    return m;
}

// van Driest wall damping of tauSGS (damping 2), the branch kernel.cl:2178-2197 keeps in
// comments beside the Fluent factor: y+ solves the log law y+ ln(E y+) = kappa U y / nu by
// Newton's method from y+ = 1 (stop when a step moves y+ by 1e-3 or less, or after 10
// steps; from y+ = 1 every iterate stays above 1/E, where 1 + ln(E y+) > 0), and the factor
// is min(1, (kappa / Cs)(1 + 1e-10 - exp(-y+ / A+)) y)^2, A+ = 26, E = 9.8,
// nu = (tau - 1/2) / 3.
template <typename Real>
__device__ inline Real van_driest(Real tau, Real U, Real y, Real Cs)
{
    const Real kappa = Real(0.41), Aplus = Real(26), E = Real(9.8);
    const Real nu = (tau - Real(0.5)) / Real(3);
    Real yp = Real(1), ypn;
    int it = 0;
    do {
        ypn = yp;
        yp = ((kappa * U * y / nu) + yp) / (Real(1) + log(E * yp));
        it++;
    } while (fabs(yp - ypn) > Real(0.001) && it < 10);
    const Real d = fmin(Real(1), (kappa / Cs) * ((Real(1) + Real(1e-10)) - exp(-yp / Aplus)) * y);
    return d * d;
}

// kernel.cl:2133-2201 smagorinskyTauSGS.  The reference sums c_a c_b (f_q - feq_q) over q
// with the incompressible feq (rho + 3 c.u + 4.5 (c.u)^2 - 1.5 u^2) w_q, whose second
// moment is rho/3 delta_ab + u_a u_b; Pi_neq is formed from the shared moments instead.
template <typename Real>
__device__ inline Real smagorinsky_tau(const Mom19<Real> &m, Real u, Real v, Real w, Real tau, Real inv_rho,
                                       Real LES, Real sdf, Real Cs, int damping)
{
    const Real r3 = m.rho * (Real(1) / Real(3));
    const Real Pxx = m.sxx - r3 - u * u, Pyy = m.syy - r3 - v * v, Pzz = m.szz - r3 - w * w;
    const Real Pxy = m.sxy - u * v, Pxz = m.sxz - u * w, Pyz = m.syz - v * w;
    const Real PP = fsqrt(Pxx * Pxx + Pyy * Pyy + Pzz * Pzz + Real(2) * (Pxy * Pxy + Pxz * Pxz + Pyz * Pyz));
    Real t = LES * Real(0.5) *
             (-tau + fsqrt(tau * tau + Real(18) * Real(1.4142135623730951) * Cs * Cs * PP * inv_rho));
    if (damping == 1 && sdf != Real(10000) && sdf > Real(0)) {
        const Real d = fmin(Real(1), Real(0.41) * sdf / Cs);
        t *= d * d;
    } else if (damping == 2 && sdf != Real(10000) && sdf > Real(0)) {
        t *= van_driest<Real>(tau, sqrt(u * u + v * v + w * w), sdf, Cs);
    }
    return t;
}

// kernel.cl:2444-2503 tauSpongeZone
template <typename Real, int Q>
__device__ inline Real sponge_tau(const StepArgs<Real, Q> &a, Real tau, Real tauSGS, int i, int j, int k)
{
    const Real spz = a.spz;
    const int m = a.sponge_mask;
    if (m == 0) return tau;
    const Real one_m = Real(1) - tauSGS;
    if ((m & 1) && Real(i) < Real(a.nx) * spz) {
        const Real fx = Real(i) * a.inv_spx;
        tau = (Real(1) - fx) * one_m + fx * tau;
    }
    if ((m & 2) && Real(i) > Real(a.nx) * (Real(1) - spz)) {
        const Real fx = Real(a.nx - i) * a.inv_spx;
        tau = (Real(1) - fx) * one_m + fx * tau;
    }
    if ((m & 4) && Real(j) < Real(a.ny) * spz) {
        const Real fx = Real(j) * a.inv_spy;
        tau = (Real(1) - fx) * one_m + fx * tau;
    }
    if ((m & 8) && Real(j) > Real(a.ny) * (Real(1) - spz)) {
        const Real fx = Real(a.ny - j) * a.inv_spy;
        tau = (Real(1) - fx) * one_m + fx * tau;
    }
    if ((m & 16) && Real(k) < Real(a.nz) * spz) {
        const Real fx = Real(k) * a.inv_spz;
        tau = (Real(1) - fx) * one_m + fx * tau;
    }
    if ((m & 32) && Real(k) > Real(a.nz) * (Real(1) - spz)) {
        const Real fx = Real(a.nz - k) * a.inv_spz;
        tau = (Real(1) - fx) * one_m + fx * tau;
    }
    return tau;
}

// kernel.cl:3156-3309 recursive-regularized collision (bulk/shear split of the
// 2nd-order non-equilibrium moments, 3rd/4th order rebuilt recursively), with the
// body force S_q = rho w_q 3 c_qx dpdx.  u is the force-shifted velocity.
template <typename Real>
__device__ inline void collide_rr(Real *out, const Mom19<Real> &m, Real inv_rho, Real u, Real v, Real w,
                                  Real omegaEff, Real omegaB, Real dpdx)
{
    const Real cs2 = Real(1) / Real(3), cs4 = Real(1) / Real(9);
    const Real rho = m.rho;
    // second-order Hermite moments of ft per unit density
    const Real R200 = (m.sxx - cs2 * rho) * inv_rho;
    const Real R020 = (m.syy - cs2 * rho) * inv_rho;
    const Real R002 = (m.szz - cs2 * rho) * inv_rho;
    const Real R110 = m.sxy * inv_rho;
    const Real R101 = m.sxz * inv_rho;
    const Real R011 = m.syz * inv_rho;

    const Real E200 = u * u, E020 = v * v, E002 = w * w, E110 = u * v, E101 = u * w, E011 = v * w;
    const Real N200 = R200 - E200, N020 = R020 - E020, N002 = R002 - E002;
    const Real N110 = R110 - E110, N101 = R101 - E101, N011 = R011 - E011;
    const Real N210 = v * N200 + Real(2) * u * N110;
    const Real N201 = w * N200 + Real(2) * u * N101;
    const Real N021 = w * N020 + Real(2) * v * N011;
    const Real N120 = u * N020 + Real(2) * v * N110;
    const Real N102 = u * N002 + Real(2) * w * N101;
    const Real N012 = v * N002 + Real(2) * w * N011;
    const Real N220 = E020 * N200 + E200 * N020 + Real(4) * E110 * N110;
    const Real N202 = E002 * N200 + E200 * N002 + Real(4) * E101 * N101;
    const Real N022 = E002 * N020 + E020 * N002 + Real(4) * E011 * N011;

    const Real omegaM = (omegaB - omegaEff) * cs2;
    const Real omegaP = omegaM + omegaEff;
    const Real C200 = R200 - omegaP * N200 - omegaM * N020 - omegaM * N002;
    const Real C020 = R020 - omegaM * N200 - omegaP * N020 - omegaM * N002;
    const Real C002 = R002 - omegaM * N200 - omegaM * N020 - omegaP * N002;
    const Real C110 = R110 - omegaEff * N110;
    const Real C101 = R101 - omegaEff * N101;
    const Real C011 = R011 - omegaEff * N011;
    const Real om1 = Real(1) - omegaEff;
    const Real M210 = E200 * v + om1 * N210 + cs2 * v;
    const Real M201 = E200 * w + om1 * N201 + cs2 * w;
    const Real M021 = E020 * w + om1 * N021 + cs2 * w;
    const Real M120 = E020 * u + om1 * N120 + cs2 * u;
    const Real M102 = E002 * u + om1 * N102 + cs2 * u;
    const Real M012 = E002 * v + om1 * N012 + cs2 * v;
    const Real M220 = E200 * E020 + om1 * N220 + cs2 * (C200 + C020) + cs4;
    const Real M202 = E200 * E002 + om1 * N202 + cs2 * (C200 + C002) + cs4;
    const Real M022 = E020 * E002 + om1 * N022 + cs2 * (C020 + C002) + cs4;
    const Real M200 = C200 + cs2, M020 = C020 + cs2, M002 = C002 + cs2;
    const Real M110 = C110, M101 = C101, M011 = C011;

    const Real h = Real(0.5) * rho, qr = Real(0.25) * rho;
    const Real F1 = rho * w19<Real>(1) * Real(3) * dpdx;   // force on axis directions
    const Real F7 = rho * w19<Real>(7) * Real(3) * dpdx;   // force on diagonals
    const Real ax = h * (u + M200 - M120 - M102 - M220 - M202);
    const Real ay = h * (v + M020 - M210 - M012 - M220 - M022);
    const Real az = h * (w + M002 - M201 - M021 - M202 - M022);
    out[0] = rho * (Real(1) - M200 - M020 - M002 + M220 + M202 + M022);
    out[1] = ax + F1;
    out[2] = rho * (-u + M120 + M102) + ax - F1;
    out[3] = ay;
    out[4] = rho * (-v + M210 + M012) + ay;
    out[5] = az;
    out[6] = rho * (-w + M201 + M021) + az;
    const Real dxy = qr * (M110 + M210 + M120 + M220);
    const Real dxz = qr * (M101 + M201 + M102 + M202);
    const Real dyz = qr * (M011 + M021 + M012 + M022);
    out[7] = dxy + F7;
    out[8] = h * (-M210 - M120) + dxy - F7;
    out[9] = h * (-M110 - M210) + dxy + F7;
    out[10] = h * (-M110 - M120) + dxy - F7;
    out[11] = dxz + F7;
    out[12] = h * (-M201 - M102) + dxz - F7;
    out[13] = h * (-M101 - M201) + dxz + F7;
    out[14] = h * (-M101 - M102) + dxz - F7;
    out[15] = dyz;
    out[16] = h * (-M021 - M012) + dyz;
    out[17] = h * (-M011 - M021) + dyz;
    out[18] = h * (-M011 - M012) + dyz;
}

// The populations that enter through an outlet face, from the cell's and the inner
// neighbour's own (previous) values: direction q at the min face, its opposite at the max
// face (the two ends of an axis differ: a z outlet on a 2-D lattice is refused).  One select
// of the direction per pair, so that the ten loads go out together.
template <int DIR, typename S, typename Real>
__device__ __forceinline__ void outlet19(Real *ft, const S *fs, uint32_t fstride, long ic, bool lo, long st, Real s)
{
    const uint32_t inner = (uint32_t)(lo ? ic + st : ic - st);
    S fi[19], fc[19];
#pragma unroll
    for (int q = 1; q < 19; q++) {
        if ((DIR == 0 ? L19::cx[q] : (DIR == 1 ? L19::cy[q] : L19::cz[q])) != 1) continue;
        const int qd = lo ? q : L19::opp(q);
        fi[q] = fs[pop_at<19, S>(qd, inner, fstride)];
        fc[q] = fs[pop_at<19, S>(qd, (uint32_t)ic, fstride)];
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int q = 1; q < 19; q++) {
        if ((DIR == 0 ? L19::cx[q] : (DIR == 1 ? L19::cy[q] : L19::cz[q])) != 1) continue;
        const int qo = L19::opp(q);
        const Real v = s * Codec<S, Real, 19>::load(&fi[q], q, w19<Real>(q)) +
                       (Real(1) - s) * Codec<S, Real, 19>::load(&fc[q], q, w19<Real>(q));
        ft[q] = pick(lo, v, ft[q]);
        ft[qo] = pick(lo, ft[qo], v);
    }
}

// Boundary handling of a domain-face cell: streaming with walls, then the face
// conditions in the reference's order (kernel.cl:3581-3592).
// xonly = false: every direction is streamed here.  xonly = true: a cell on an x face (and
// on no other face) whose directions were pulled from the interior offsets already; only
// the directions that cross its face (c_x = +1 at i = 0, c_x = -1 at i = nx - 1) are
// streamed again.  The face conditions follow in either case.
// early: the face velocity, where it has been loaded already (else null).
template <typename S, typename Real, typename E>
__device__ __forceinline__ void face_cell(const Step19Args<Real> &a, Real *ft, uint32_t fl, long ic, int i, int j, int k,
                                       Real omega, bool xonly, const E *early)
{
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const S *fs = (const S *)a.fsrc;
    const int b1 = flag_code(fl, F_B1_SHIFT), b2 = flag_code(fl, F_B2_SHIFT), b3 = flag_code(fl, F_B3_SHIFT);
    const int xs = (i == 0) ? 1 : -1;
    // Every direction has exactly one source -- the upwind cell, or across a wall the cell's own
    // reflected slot -- so its address is selected and all loads go out together.  A branch
    // per direction with a load in either arm made a face wave wait for memory 18 times in a
    // row, which bounds small lattices: with the velocity gradient of wale_tau likewise, a
    // 32^3 FP32 cavity went from 14.5 to 9.8 us per step, 64^3 FP64 from 27.5 to 20 us, 60
    // FP16 lattices of edge 24-96 from 0.81 to 0.70 ms.
    S raw[19];
    if (!xonly) {
        // (each address right before its load: computed ahead of the loads, 18 64-bit addresses
        // would not fit the registers beside the populations)
        raw[0] = fs[pop_at<19, S>(0, (uint32_t)ic, a.fstride)];
#pragma unroll
        for (int q = 1; q < 19; q++) {
            const long src = face_upwind(q, ic, i, j, k, nx, ny, nz, b1, b2, b3);
            const size_t own = pop_at<19, S>(mirror_q(q, b1, b2, b3), (uint32_t)ic, a.fstride);
            const size_t up = pop_at<19, S>(q, (uint32_t)src, a.fstride);
            raw[q] = fs[src < 0 ? own : up];
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int q = 0; q < 19; q++) ft[q] = Codec<S, Real, 19>::load(&raw[q], q, w19<Real>(q));
    } else {
        // the five directions that cross the cell's x face: q with c_x = +1 at i = 0, its
        // opposite at i = nx - 1 (j and k are interior: no other face is crossed)
        const bool lo = (xs == 1), wall = is_wall_code(b1);
#pragma unroll
        for (int q = 1; q < 19; q++) {
            if (L19::cx[q] != 1) continue;
            const int qo = L19::opp(q);
            const uint32_t src = (uint32_t)(ic - (lo ? a.off[q] : a.off[qo]) + xs * nx);
            const int qb = lo ? mirror_q(q, b1, b2, b3) : mirror_q(qo, b1, b2, b3);
            const size_t own = pop_at<19, S>(qb, (uint32_t)ic, a.fstride);
            const size_t up = pop_at<19, S>(lo ? q : qo, src, a.fstride);
            raw[q] = fs[wall ? own : up];
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int q = 1; q < 19; q++) {
            if (L19::cx[q] != 1) continue;
            const Real v = Codec<S, Real, 19>::load(&raw[q], q, w19<Real>(q));
            ft[q] = pick(lo, v, ft[q]);
            ft[L19::opp(q)] = pick(lo, ft[L19::opp(q)], v);
        }
    }
    const int corner = corner_flag(b3, i, j, k, nx, ny, nz);
    const long sy = nx, sz = (long)nx * ny;

    // fixedVelocityBC, kernel.cl:1397-1512
    if (corner == 0 && (b1 == BC_FIXEDVELOCITY || b2 == BC_FIXEDVELOCITY || b3 == BC_FIXEDVELOCITY)) {
        const Real u0 = early ? early->u0 : a.u0[ic], v0 = early ? early->v0 : a.v0[ic],
                   w0 = early ? early->w0 : a.w0[ic];
        if (b1 == BC_FIXEDVELOCITY && (i == 0 || i == nx - 1)) {
            const bool lo = (i == 0);
            Real rhow = zouhe_sum(ft, 0, lo) / (lo ? Real(1) - u0 : Real(1) + u0);
            if (lo && u0 < Real(0)) rhow = a.rho_o[ic + 1];
            if (!lo && u0 > Real(0)) rhow = a.rho_o[ic];  // own stored density (K19:1424-1428)
            ladd(ft, 0, lo, rhow, u0, v0, w0);
        }
        if (b2 == BC_FIXEDVELOCITY && (j == 0 || j == ny - 1)) {
            const bool lo = (j == 0);
            Real rhow = zouhe_sum(ft, 1, lo) / (lo ? Real(1) - v0 : Real(1) + v0);
            if (lo && v0 < Real(0)) rhow = a.rho_o[ic + sy];
            if (!lo && v0 > Real(0)) rhow = a.rho_o[ic - sy];
            ladd(ft, 1, lo, rhow, v0, u0, w0);
        }
        if (b3 == BC_FIXEDVELOCITY && (k == 0 || k == nz - 1)) {
            const bool lo = (k == 0);
            Real rhow = zouhe_sum(ft, 2, lo) / (lo ? Real(1) - w0 : Real(1) + w0);
            if (lo && w0 < Real(0)) rhow = a.rho_o[ic + sz];
            if (!lo && w0 > Real(0)) rhow = a.rho_o[ic - sz];
            ladd(ft, 2, lo, rhow, w0, u0, v0);
        }
    }

    // fixedDensityBC with rho_w = 1, kernel.cl:1514-1611
    if (corner == 0 && (b1 == BC_FIXEDDENSITY || b2 == BC_FIXEDDENSITY || b3 == BC_FIXEDDENSITY)) {
        const Real uc = a.u_o[ic], vc = a.v_o[ic], wc = a.w_o[ic];
#pragma unroll
        for (int dir = 0; dir < 3; dir++) {
            const int code = dir == 0 ? b1 : (dir == 1 ? b2 : b3);
            if (code != BC_FIXEDDENSITY) continue;
            const int pos = dir == 0 ? i : (dir == 1 ? j : k);
            const int n = dir == 0 ? nx : (dir == 1 ? ny : nz);
            const long st = dir == 0 ? 1 : (dir == 1 ? sy : sz);
            // inner neighbour: index 1 at the min face, n-2 otherwise (kernel.cl:1520, 1560, 1590)
            const long inner = (pos == 0) ? ic + st : ic + (long)(n - 2 - pos) * st;
            const Real ue = uc + Real(0.5) * (uc - a.u_o[inner]);
            const Real ve = vc + Real(0.5) * (vc - a.v_o[inner]);
            const Real we = wc + Real(0.5) * (wc - a.w_o[inner]);
            const Real uSqr = ue * ue + ve * ve + we * we;
            const bool atlo = (pos == 0), athi = (pos == n - 1);
#pragma unroll
            for (int q = 1; q < 19; q++) {
                const int cn = dir == 0 ? L19::cx[q] : (dir == 1 ? L19::cy[q] : L19::cz[q]);
                if ((atlo && cn == 1) || (athi && cn == -1)) {
                    const Real uDotC = ue * Real(L19::cx[q]) + ve * Real(L19::cy[q]) + we * Real(L19::cz[q]);
                    ft[q] = -ft[q] + Real(2) * w19<Real>(q) * Real(1)
                                         * (Real(1) + Real(4.5) * uDotC * uDotC - Real(1.5) * uSqr);
                }
            }
        }
    }

    // wallFunctionBC, kernel.cl:1654-1924 (stationary wall, tangential slip velocity)
    if (corner == 0 && (b1 == BC_WALLFUNCTION || b2 == BC_WALLFUNCTION || b3 == BC_WALLFUNCTION)) {
        const Real nu = (Real(1) / omega - Real(0.5)) / Real(3);
        // wall momentum of this step's domain-face links (off the corners a cell lies on one
        // wall face, so no condition above has changed these populations)
        Real Fx = 0, Fy = 0, Fz = 0;
#pragma unroll
        for (int q = 1; q < 19; q++)
            if (face_upwind(q, ic, i, j, k, nx, ny, nz, b1, b2, b3) < 0) {
                Fx += Real(-2) * ft[q] * Real(L19::cx[q]);
                Fy += Real(-2) * ft[q] * Real(L19::cy[q]);
                Fz += Real(-2) * ft[q] * Real(L19::cz[q]);
            }
#pragma unroll
        for (int dir = 0; dir < 3; dir++) {
            const int code = dir == 0 ? b1 : (dir == 1 ? b2 : b3);
            const int pos = dir == 0 ? i : (dir == 1 ? j : k);
            const int n = dir == 0 ? nx : (dir == 1 ? ny : nz);
            if (code != BC_WALLFUNCTION || !(pos == 0 || pos == n - 1)) continue;
            const bool lo = (pos == 0);
            const long st = dir == 0 ? 1 : (dir == 1 ? sy : sz);
            const Real rhow = zouhe_sum(ft, dir, lo);
            // neighbour sampled for the wall law: the next cell inward; the z faces of a
            // 2-D lattice sample the cell itself (K19:1848)
            long nb = lo ? ic + st : ic - st;
            if (dir == 2) nb = (nz - 1 != 0) ? ic + st : ic;
            const Real *t1 = dir == 0 ? a.v_o : a.u_o;
            const Real *t2 = dir == 2 ? a.v_o : a.w_o;
            Real p = t1[nb], s = t2[nb];
            Real magUp = sqrt(p * p + s * s);
            Real ut1 = 0, ut2 = 0;
            if (magUp != Real(0)) {
                const Real tauw = calc_tauw<Real>(rhow, magUp, nu);
                p = t1[ic];
                s = t2[ic];
                magUp = sqrt(p * p + s * s);
                if ((dir == 2 && lo) || magUp != Real(0)) {
                    const Real e1 = p / magUp, e2 = s / magUp;
                    const Real Fw1 = dir == 0 ? Fy : Fx;
                    const Real Fw2 = dir == 2 ? Fy : Fz;
                    ut1 = Real(-3) * (tauw * e1 - Fw1) / rhow;
                    ut2 = Real(-3) * (tauw * e2 - Fw2) / rhow;
                }
            }
            ladd(ft, dir, lo, rhow, Real(0), ut1, ut2);
        }
    }

    // outflowBC, kernel.cl:2005-2097: convective outlet with the cell's last velocity
    if (b1 == BC_OUTLET || b2 == BC_OUTLET || b3 == BC_OUTLET) {
        const Real is3 = Real(0.57735026918962576);
        if (b1 == BC_OUTLET && (i == 0 || i == nx - 1)) outlet19<0, S>(ft, fs, a.fstride, ic, i == 0, 1, is3 - a.u_o[ic]);
        if (b2 == BC_OUTLET && (j == 0 || j == ny - 1)) outlet19<1, S>(ft, fs, a.fstride, ic, j == 0, sy, is3 - a.v_o[ic]);
        if (b3 == BC_OUTLET && (k == 0 || k == nz - 1)) outlet19<2, S>(ft, fs, a.fstride, ic, k == 0, sz, is3 - a.w_o[ic]);
    }
}

// The face conditions of a cell on an x face and no other (an XMIX wave's), its directions pulled
// from the interior offsets already, for the face codes FixedVelocity and Outlet; false, and
// nothing done, for the others and where a Symmetry code mirrors.  The five directions that
// cross the face take the cell's own reversed slot (fixed velocity) or the inner neighbour's value
// beside the cell's own (outlet), and the face's velocity or rate is loaded with them: one
// trip to memory.  In the general path the streaming, the velocity, the outlet's rate and its
// populations were four trips and some 300 instructions for the one or two face cells of a
// wave.  The formulas are face_cell's, in its order of operations.  60 FP16 lattices of edge
// 24-96, half of them channels: 0.70 -> 0.65 ms per step; FP16 backstep 289 -> 280 us.  (Walls and periodic faces stay with
// the cell body's own shortcut: folded into this one, their waves ran 2 % slower.)
template <typename S, typename Real>
__device__ __forceinline__ bool x_face19(const Step19Args<Real> &a, Real *ft, uint32_t fl, uint32_t ic, int i)
{
    const int b1 = flag_code(fl, F_B1_SHIFT), b2 = flag_code(fl, F_B2_SHIFT), b3 = flag_code(fl, F_B3_SHIFT);
    const bool fixed = b1 == BC_FIXEDVELOCITY;
    if (!(fixed || b1 == BC_OUTLET) || b2 == BC_SYMMETRY || b3 == BC_SYMMETRY) return false;
    const S *fs = (const S *)a.fsrc;
    const bool lo = (i == 0);
    // fixed: the wall velocity; outlet: the cell's last x velocity
    const Real u = fixed ? a.u0[ic] : a.u_o[ic];
    const uint32_t src = fixed ? ic : (lo ? ic + 1u : ic - 1u);
    S ra[19], rb[19];
#pragma unroll
    for (int q = 1; q < 19; q++) {
        if (L19::cx[q] != 1) continue;
        const int qo = L19::opp(q);
        ra[q] = fs[pop_at<19, S>(lo == fixed ? qo : q, src, a.fstride)];
        rb[q] = fs[pop_at<19, S>(lo ? q : qo, ic, a.fstride)];
        __builtin_amdgcn_sched_barrier(0);
    }
    const Real s = Real(0.57735026918962576) - u;
#pragma unroll
    for (int q = 1; q < 19; q++) {
        if (L19::cx[q] != 1) continue;
        const int qo = L19::opp(q);
        const Real fi = Codec<S, Real, 19>::load(&ra[q], q, w19<Real>(q));
        const Real fc = Codec<S, Real, 19>::load(&rb[q], q, w19<Real>(q));
        const Real vo = s * fi + (Real(1) - s) * fc;
        const Real v = pick(fixed, fi, vo);
        ft[q] = pick(lo, v, ft[q]);
        ft[qo] = pick(lo, ft[qo], v);
    }
    if (fixed) {
        Real rhow = zouhe_sum(ft, 0, lo) / (lo ? Real(1) - u : Real(1) + u);
        if (lo && u < Real(0)) rhow = a.rho_o[ic + 1];
        if (!lo && u > Real(0)) rhow = a.rho_o[ic];  // own stored density (K19:1424-1428)
        ladd(ft, 0, lo, rhow, u, a.v0[ic], a.w0[ic]);
    }
    return true;
}

// IBB selects the interpolated bounce-back at compile time: its loop adds registers to the
// whole kernel, which the kernels without it should not carry.  AA: 0 two-lattice streaming, 1 and 2
// the two half-steps of in-place streaming (the cell body describes them).  PASS: 0 every
// cell; 1 every cell but the lattice-face cells; 2 the face cells of the list a.fcells.  A
// wave that holds face and interior cells runs both the face path and the interior pull;
// two passes keep them apart (TUNE_SPLIT runs 1 then 2; both read only the previous
// step's arrays).  It pays where such waves are many and the step is bound by instruction
// issue, and costs a second launch's drain where the step is bound by HBM.
// PASS 3 runs both passes in one grid: the first face_blocks(a) work-groups take the face
// cells of the list, the others the cells off the faces, so that no wave runs both paths
// and no second launch waits for the first to drain (the face work-groups are dispatched
// first and run beside the interior ones).
// (rounded up to a multiple of 8, so that the blocks after them keep their hardware XCD
// order; the work-groups past the list end at once)
// PASS 4 runs every cell as 0 does, in the form for small lattices (kLatencyCells).
template <typename A>
__device__ inline uint32_t face_blocks(const A &a)
{
    return merged_face_blocks(a.nface, blockDim.x);
}

// PASS 4 is the form for lattices whose waves are all resident at once and which wait for memory
// one trip after another (kLatencyCells): it reads its arguments' cache lines together, then the
// flags, the face velocity and WALE's neighbours beside the wave's class, where the others load
// each when the one before has said that it is needed.  32^3 cavity 10.0 -> 8.3 us per step in
// FP32, 11.2 -> 9.3 FP64, 9.4 -> 7.8 FP16 (a step that only streams, 2.7); of the 1.7 us, WALE's trip is 1.1.
// Its registers (82 FP32, 146 FP64) cost occupancy, so that it ends where the waves no longer
// fit: three waves per SIMD in FP32 (58^3 13.3 -> 11.5 us, but 64^3 13.1 -> 13.6), four with 16-bit
// values (64^3 14.2 -> 12.4, 72^3 15.7 -> 19.1), one in FP64 (40^3 11.4 -> 9.8, the 192x24x24
// box 11.5 -> 11.8).  D3Q27 gains a tenth in a cavity and loses a twentieth in a periodic box: it
// has no such form.
template <typename S>
constexpr uint32_t kLatencyCells = 1024u * 64u * (sizeof(S) == 8 ? 1u : (sizeof(S) == 4 ? 3u : 4u));

// Waves per SIMD the step kernel is held to: eight (64 VGPRs), which the compiler reaches
// without spilling by interleaving each direction's pull address with its load; seven with
// the interpolated bounce-back, whose groups of links spill at eight; FP64 and the latency form as
// the compiler chooses.
template <typename S, typename Real, int SGS, bool IBB, int PASS>
constexpr int kStep19MinWaves = (sizeof(Real) == 8 || PASS == 4) ? 1 : (IBB ? 7 : 8);

// reads one word of every 64 bytes of the launch arguments: the scalar loads that take them
// where they are used then find them in the scalar cache, instead of missing it once per line
// along the kernel (0.4 us of a small lattice's step; 400x160x16 cylinder with the interpolated
// bounce-back, FP32: 37.9 -> 37.2 us; no gain in its 16-bit form or on large lattices)
template <typename A>
__device__ __forceinline__ void touch_args()
{
    typedef const __attribute__((address_space(4))) uint32_t const_u32;
    const_u32 *p = (const_u32 *)__builtin_amdgcn_kernarg_segment_ptr();
    uint32_t x = 0;
#pragma unroll
    for (size_t i = 0; i < sizeof(A) / 4; i += 16) x |= p[i];
    asm volatile("" ::"s"(x));
}

template <typename S, typename Real, int SGS, bool IBB = false, int AA = 0, int PASS = 0>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kStep19MinWaves<S, Real, SGS, IBB, PASS>, 8)))
step19_kernel(const Step19Args<Real> a)
{
    // (and FP32 with the interpolated bounce-back, whose waves along a wall are as serial)
    if constexpr (PASS == 4 || (IBB && PASS == 0 && sizeof(S) == 4)) touch_args<Step19Args<Real>>();
    const uint32_t nfb = (PASS == 3) ? face_blocks(a) : 0u;
    const bool face_wg = (PASS == 2) || (PASS == 3 && blockIdx.x < nfb);
    uint32_t icu;
    if (face_wg) {
        const uint32_t lin = blockIdx.x * blockDim.x + threadIdx.x;
        if (lin >= a.nface) return;
        icu = a.fcells[lin];
        if (face_pass_skips(cell_wave_class(a.wclass, icu))) return;
    } else {
        const uint32_t g = blockIdx.x - nfb;
        const uint32_t blk = ordered_block(g, gridDim.x - nfb, a.tune);
        const uint32_t lin = blk * blockDim.x + threadIdx.x;
        if (lin >= a.N) return;
        icu = (a.tune & TUNE_YTILE) ? ytile_cell(a, lin) : lin;
    }
#define CELL_RETURN return
#define CELL_IBB IBB
#define CELL_WALE_INTERIOR true
#define CELL_AA AA
#define CELL_SKIP_FACE (PASS == 1 || (PASS == 3 && !face_wg))
#define CELL_PURE_OK (AA == 0 && !face_wg)
#define CELL_ALIGNED (!face_wg && a.wave_runs)
#define CELL_KEEP a.keep
#define CELL_EARLY (PASS == 4)
#include "d3q19_cell.inc"
#undef CELL_EARLY
#undef CELL_KEEP
#undef CELL_ALIGNED
#undef CELL_PURE_OK
#undef CELL_SKIP_FACE
#undef CELL_AA
#undef CELL_WALE_INTERIOR
#undef CELL_IBB
#undef CELL_RETURN
}

// In-place streaming: after the first half-step, out[p] of cell x sits in slot opp(p) of
// x + c_p and out[opp(p)] of x + c_p in slot p of x, for every link between two fluid cells
// that is not a wall link.  Exchanging the two restores the two-lattice layout (and
// exchanging again undoes it); cell x exchanges its odd directions p (opp(p) = p + 1), so
// every pair is exchanged once.  Links across a wall or to a solid cell already hold their
// value in the cell's own slot p.
template <typename S>
__global__ void aa_swap19_kernel(uint32_t N, int nx, int ny, int nz, FastDiv dnx, FastDiv dny,
                                 const uint16_t *__restrict__ flag, size_t FS, S *f)
{
    const uint32_t icu = blockIdx.x * blockDim.x + threadIdx.x;
    if (icu >= N) return;
    const uint32_t fl = flag[icu];
    if (fl & F_SOLID) return;
    const uint32_t t = fdiv(icu, dnx);
    const int i = (int)(icu - t * (uint32_t)nx);
    const uint32_t kk = fdiv(t, dny);
    const int j = (int)(t - kk * (uint32_t)ny);
    const int k = (int)kk;
    const int b1 = flag_code(fl, F_B1_SHIFT), b2 = flag_code(fl, F_B2_SHIFT), b3 = flag_code(fl, F_B3_SHIFT);
    const long sy = nx, sz = (nz == 1) ? 0 : (long)nx * ny;
#pragma unroll
    for (int p = 1; p < 19; p += 2) {
        const int po = p + 1;
        // the cell x + c_p: the pull source of direction opp(p)
        const long nb = (fl & F_FACE) ? face_upwind(po, (long)icu, i, j, k, nx, ny, nz, b1, b2, b3)
                                      : (long)icu + L19::cx[p] + L19::cy[p] * sy + L19::cz[p] * sz;
        if (nb < 0 || (flag[nb] & F_SOLID)) continue;
        S *x = f + pop_at<19, S>(p, icu, FS);
        S *y = f + pop_at<19, S>(po, (uint32_t)nb, FS);
        const S tx = *x;
        *x = *y;
        *y = tx;
    }
}

}  // namespace lbffs
