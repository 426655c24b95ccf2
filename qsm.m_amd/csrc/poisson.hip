// poisson.hip -- multigrid-preconditioned CG for the masked Poisson problem
// (src/utils/poisson_solver/mgpcg.m, mex/mgpcg_mex.c) and Laplacian phase
// unwrapping (src/unwrap/unwrapLaplacian.m) on gfx950.
//
// The system (lapmg_mex.c): on the voxels of the mask G, -Lap_h v = f with
// the 7-point Laplacian, v = 0 off the mask and on a one-voxel border added
// around the volume (mgpcg_mex.c: mx_pad_boundary).  PCG (mgpcg_mex.c:
// mx_pcg) stops when ||r|| <= tol ||f|| or after maxit iterations; its
// preconditioner is mgopts.maxit V-cycles (mx_mg, mx_cycle): pre-smoothing
// on G and on the boundary band B (2^l nboundary sweeps on level l, from
// per-colour index lists of the band), the residual, full-weighting
// restriction onto the coarse mask, the coarse cycle, trilinear
// correction, the mirrored post-smoothing; on the
// coarsest level the reference sweeps to a relative residual of 1e-8.
// The grid hierarchy (the voxel size doubles per level), the masks (a coarse
// voxel is active iff its 8 fine children are: coarsen_grid_mex.c), the
// band (boundary_mask_mex.c) and the transfer weights (restrict_mex.c,
// correct_mex.c) are the reference's.  The smoother is red-black
// Gauss-Seidel (the reference's GAUSS_SEIDEL_RED_BLACK variant) with the
// reference's colour order in its reverse sweeps (gauss_seidel_mex.c:
// 141-163: the first colour there is the one of parity nx + 1).  Two
// choices differ from the reference and change only the preconditioner,
// hence how fast PCG converges, not what it converges to: every voxel of a
// colour is updated (the reference's loops skip the row end of the second
// colour on rows with j = k mod 2, which on a mask that touches the
// volume's faces makes the V-cycle a poor preconditioner), and the coarsest
// level takes a fixed-degree Chebyshev iteration on the Jacobi-scaled
// operator instead of rounds of 256 Gauss-Seidel sweeps.  Its degree
// reduces the coarse error by 1e3 over the spectrum bound of the level's
// box (the masked operator is a principal submatrix of the box's, so the
// bound holds for any mask); its steps are stencil updates by many
// workgroups, with no reduction, four steps per launch on small levels and
// one on large ones, and a fixed polynomial keeps the V-cycle a fixed linear
// map, as PCG requires of its preconditioner.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "common.h"

using namespace qsm;

namespace {

constexpr int BX = 64, BY = 4, NT = BX * BY;
constexpr int MAX_LEVELS = 16;    // at most 16 grid levels (mgpcg_mex.c: MAX_DEPTH)
constexpr int CHEB_MAX = 512;     // Chebyshev degree cap on the coarsest level
constexpr double CHEB_EPS = 1e-3; // coarse error reduction it aims for
constexpr int DOT_BLOCKS = 1024;  // fixed grid of the dot products

// A grid and its storage.  Every field of the solver is kept split by colour
// (the parity of i + j + k): colour c's voxels of row (j, k) lie together,
// voxel i = 2 t + ((c + j + k) & 1) at position t + P (j + ny k) of colour
// c's half, P the half row rounded up to a multiple of four.  A red-black
// pass then reads and writes whole cache lines of what it needs -- one
// colour of f, the mask and v, the other colour of v -- where the natural
// order drags both colours of all three through every pass (at 258x258x178
// padded, FP32: 77 MB against 153 MB; a pass 37.4 -> 13.8 us).  At equal t a voxel's y and z
// neighbours stand at the same t of the other colour, its x neighbours at
// t - 1 and t (parity 0) or t and t + 1 (parity 1).  Positions past the row's
// end are zero and their mask bytes clear.
struct Dim {
    int nx, ny, nz;
    int P;
    __host__ __device__ size_t rows() const { return size_t(ny) * nz; }
    __host__ __device__ size_t half() const { return P * rows(); }   // positions per colour
    __host__ __device__ size_t n() const { return 2 * half(); }
    __host__ __device__ size_t nat() const { return nx * rows(); }   // natural order
    // position of voxel (i, j, k)
    __host__ __device__ size_t at(int i, int j, int k) const
    {
        return size_t((i + j + k) & 1) * half() + size_t(i >> 1) +
               size_t(P) * (size_t(j) + size_t(ny) * k);
    }
};

Dim make_dim(int nx, int ny, int nz) { return Dim{nx, ny, nz, ((nx + 1) / 2 + 3) / 4 * 4}; }

// one lane per voxel of the natural grid
dim3 grid3(Dim d) { return dim3((d.nx + BX - 1) / BX, (d.ny + BY - 1) / BY, d.nz); }

// one lane per four positions of a colour's plane
dim3 grid4(Dim d, int colours)
{
    return dim3((unsigned(d.P / 4) * unsigned(d.ny) + NT - 1) / NT, colours, d.nz);
}

__device__ __forceinline__ bool vox(Dim d, int &i, int &j, int &k)
{
    int bx, by, bz;
    xcd_block3(bx, by, bz);  // a slab of planes per XCD
    i = bx * BX + threadIdx.x;
    j = by * BY + threadIdx.y;
    k = bz;
    return i < d.nx && j < d.ny;
}

// natural-order index
__device__ __forceinline__ size_t nidx(Dim d, int i, int j, int k)
{
    return size_t(i) + size_t(d.nx) * (size_t(j) + size_t(d.ny) * k);
}

__device__ __forceinline__ bool interior(Dim d, int i, int j, int k)
{
    return i > 0 && j > 0 && k > 0 && i < d.nx - 1 && j < d.ny - 1 && k < d.nz - 1;
}

// Four consecutive positions: one wide load or store (rows start at
// multiples of four, the fields at multiples of 256 bytes).
template <typename T>
struct alignas(4 * sizeof(T)) V4 {
    T a[4];
};

template <typename T>
__device__ __forceinline__ V4<T> ld4(const T *p) { return *reinterpret_cast<const V4<T> *>(p); }

template <typename T>
__device__ __forceinline__ void st4(T *p, const V4<T> &v) { *reinterpret_cast<V4<T> *>(p) = v; }

__device__ __forceinline__ uint32_t ldm4(const uint8_t *p)
{
    return *reinterpret_cast<const uint32_t *>(p);
}

// Group of four positions of a lane of a grid4 launch: colour c, plane k,
// first position p within the colour's half, parity b of its row.
__device__ __forceinline__ bool group4(Dim d, int &c, int &j, int &k, size_t &p, int &b)
{
    int bx, by, bz;
    xcd_block3(bx, by, bz);
    const unsigned g4 = unsigned(d.P) / 4, u = unsigned(bx) * NT + threadIdx.x;
    if (u >= g4 * unsigned(d.ny)) return false;
    c = by;
    k = bz;
    j = int(u / g4);
    p = size_t(4) * u + size_t(d.P) * d.ny * k;
    b = (c + j + k) & 1;
    return true;
}

// The six neighbours of four positions at p of parity b, o the other
// colour's half: what lies at -x, +x, -y, +y, -z, +z of each.
template <typename T>
struct Nb4 {
    V4<T> xm, xp, ym, yp, zm, zp;
};

template <typename T>
__device__ __forceinline__ void nb4(const T *o, size_t p, int b, Dim d, Nb4<T> &n)
{
    const size_t sy = size_t(d.P), sz = size_t(d.P) * d.ny;
    const V4<T> c = ld4(o + p);
    const T e = o[b ? p + 4 : p - 1];
    n.ym = ld4(o + p - sy);
    n.yp = ld4(o + p + sy);
    n.zm = ld4(o + p - sz);
    n.zp = ld4(o + p + sz);
    n.xm = b ? c : V4<T>{{e, c.a[0], c.a[1], c.a[2]}};
    n.xp = b ? V4<T>{{c.a[1], c.a[2], c.a[3], e}} : c;
}

// Laplacian coefficients as lapmg_mex.c forms them (in double): 1 / h^2 per
// axis, h the voxel size times 2^level (mgpcg_mex.c: mx_init).
struct Lap {
    double hx, hy, hz;
};

Lap lap_at(const double vsz[3], int level)
{
    const double s = std::ldexp(1.0, level);
    const double h[3] = {vsz[0] * s, vsz[1] * s, vsz[2] * s};
    return Lap{1.0 / (h[0] * h[0]), 1.0 / (h[1] * h[1]), 1.0 / (h[2] * h[2])};
}

// ---- padding -------------------------------------------------------------

// out = in with a zero border of one voxel; sgn_mask != 0: out = sgn_mask *
// mask .* in (unwrapLaplacian's -m.*d2u).  One lane per position, those past
// the row's end included.  G (may be null): the mask with a zero border, in
// natural order, here and not in a launch of its own: 15 us for both at
// 258x258x62 FP32 against 11 + 17, and a launch more ahead of the set-up's
// read-back costs the smallest solves 25 us (set-up alone 68 against 94).
template <typename T>
__global__ __launch_bounds__(NT) void pad_kernel(T *out, const T *in, uint8_t *G, const uint8_t *m,
                                                 Dim dp, T sgn_mask)
{
    int c, j, k, b;
    size_t p;
    if (!group4(dp, c, j, k, p, b)) return;
    const int t = int(p - size_t(dp.P) * (size_t(j) + size_t(dp.ny) * k));
    V4<T> v;
    for (int e = 0; e < 4; ++e) {
        const int i = 2 * (t + e) + b;
        const bool in_box = interior(dp, i, j, k);
        const size_t li = size_t(i - 1) +
                          size_t(dp.nx - 2) * (size_t(j - 1) + size_t(dp.ny - 2) * (k - 1));
        v.a[e] = T(0);
        if (in_box) v.a[e] = (sgn_mask != T(0)) ? sgn_mask * (T(m[li] ? 1 : 0) * in[li]) : in[li];
        if (G && i < dp.nx) G[nidx(dp, i, j, k)] = in_box && m[li] ? 1 : 0;
    }
    st4(out + c * dp.half() + p, v);
}

template <typename T>
__global__ __launch_bounds__(NT) void unpad_kernel(T *out, const T *in, Dim dp)
{
    int i, j, k;
    if (!vox(dp, i, j, k)) return;
    if (!interior(dp, i, j, k)) return;
    out[size_t(i - 1) + size_t(dp.nx - 2) * (size_t(j - 1) + size_t(dp.ny - 2) * (k - 1))] =
        in[dp.at(i, j, k)];
}

// ---- masks of the hierarchy ----------------------------------------------

// coarsen_grid_mex.c: coarse (i2, j2, k2) is active iff the fine voxel
// (2 i2 - 1, ...) and its +1 neighbours in x, y, z (those inside the
// interior) are all active.
__global__ __launch_bounds__(NT) void coarsen_kernel(uint8_t *G2, const uint8_t *G, Dim d2, Dim d)
{
    int i2, j2, k2;
    if (!vox(d2, i2, j2, k2)) return;
    uint8_t g = 0;
    if (interior(d2, i2, j2, k2)) {
        const int i = 2 * i2 - 1, j = 2 * j2 - 1, k = 2 * k2 - 1;
        const size_t sx = 1, sy = size_t(d.nx), sz = size_t(d.nx) * d.ny;
        const size_t l = size_t(i) + sy * (size_t(j) + size_t(d.ny) * k);
        const bool bi = !(i < d.nx - 2), bj = !(j < d.ny - 2), bk = !(k < d.nz - 2);
        g = G[l] && (bi || G[l + sx]) && (bj || G[l + sy]) && (bk || G[l + sz]) &&
            (bi || bj || G[l + sx + sy]) && (bi || bk || G[l + sx + sz]) &&
            (bj || bk || G[l + sy + sz]) && (bi || bj || bk || G[l + sx + sy + sz]);
    }
    G2[nidx(d2, i2, j2, k2)] = g;
}

// boundary_mask_mex.c, first two steps: b = G on the interior's outer
// layer, and on every 2x2x2 block (starting at odd indices) that is not
// fully active.
__global__ __launch_bounds__(NT) void band_seed_kernel(uint8_t *b, const uint8_t *G, Dim d)
{
    int i, j, k;
    if (!vox(d, i, j, k)) return;
    const size_t l = nidx(d, i, j, k);
    uint8_t v = 0;
    if (interior(d, i, j, k)) {
        if (i == 1 || j == 1 || k == 1 || i == d.nx - 2 || j == d.ny - 2 || k == d.nz - 2)
            v = G[l];
        // the block that contains (i, j, k): its corner at odd indices
        const int ic = i - ((i - 1) & 1), jc = j - ((j - 1) & 1), kc = k - ((k - 1) & 1);
        const size_t sy = size_t(d.nx), sz = size_t(d.nx) * d.ny;
        const size_t lc = size_t(ic) + sy * (size_t(jc) + size_t(d.ny) * kc);
        // the reference's block loop visits corners up to the interior's last
        // index and reads the +1 neighbours, which may be the zero border
        bool full = G[lc] && G[lc + 1] && G[lc + sy] && G[lc + sz] && G[lc + 1 + sy] &&
                    G[lc + 1 + sz] && G[lc + sy + sz] && G[lc + 1 + sy + sz];
        if (!full) v = G[l];
    }
    b[l] = v;
}

// boundary_mask_mex.c, last step: B = G .* (b or any of its 6 neighbours);
// b and G in natural order, the split copies GS of G and B written here.
__global__ __launch_bounds__(NT) void band_kernel(uint8_t *B, uint8_t *GS, const uint8_t *b,
                                                  const uint8_t *G, Dim d)
{
    int c, j, k, par;
    size_t p;
    if (!group4(d, c, j, k, p, par)) return;
    const int t = int(p - size_t(d.P) * (size_t(j) + size_t(d.ny) * k));
    const size_t sy = size_t(d.nx), sz = size_t(d.nx) * d.ny;
    uint32_t vb = 0, vg = 0;
    for (int e = 0; e < 4; ++e) {
        const int i = 2 * (t + e) + par;
        if (!interior(d, i, j, k)) continue;
        const size_t l = nidx(d, i, j, k);
        if (!G[l]) continue;
        vg |= 1u << (8 * e);
        if (b[l - sz] || b[l - sy] || b[l - 1] || b[l] || b[l + 1] || b[l + sy] || b[l + sz])
            vb |= 1u << (8 * e);
    }
    *reinterpret_cast<uint32_t *>(B + c * d.half() + p) = vb;
    *reinterpret_cast<uint32_t *>(GS + c * d.half() + p) = vg;
}

// ---- the band as index lists ---------------------------------------------
//
// The band is a thin shell, but a sweep over its mask visits the whole
// grid.  Each level's band voxels are listed once per solve, per colour, in
// increasing index order: a count per row (one wave per row of the grid),
// an exclusive scan over the rows, a fill per row.  An entry is the voxel's
// position in its colour's half and the parity of its row: 2 p + b.  A band
// sweep then takes one lane per listed voxel.  Voxels of one colour do not
// read each other, so the order within a colour does not change the result.

// One wave per row (j, k): the row's band voxels of colour 0 and 1, as
// cnt[2 row + c].
__global__ __launch_bounds__(NT) void band_count_kernel(int *cnt, const uint8_t *B, Dim d)
{
    const int lane = int(threadIdx.x) & 63;
    const int row = int(blockIdx.x) * (NT / 64) + int(threadIdx.x) / 64;
    if (row >= d.ny * d.nz) return;  // whole waves
    const uint8_t *b = B + size_t(d.P) * row;
    int c0 = 0, c1 = 0;
    for (int x0 = 0; x0 < d.P; x0 += 64) {
        const int t = x0 + lane;
        c0 += __popcll(__ballot(t < d.P && b[t]));
        c1 += __popcll(__ballot(t < d.P && b[d.half() + t]));
    }
    if (lane == 0) {
        cnt[2 * row] = c0;
        cnt[2 * row + 1] = c1;
    }
}

// One block: cnt[2 row + c] becomes the exclusive prefix over rows of
// colour c; tot[0..1] the totals.
__global__ __launch_bounds__(1024) void band_scan_kernel(int *cnt, int rows, int *tot)
{
    __shared__ int part[2][1024];
    const int t = int(threadIdx.x), per = (rows + 1023) / 1024;
    const int r0 = min(rows, t * per), r1 = min(rows, r0 + per);
    int s0 = 0, s1 = 0;
    for (int r = r0; r < r1; ++r) {
        s0 += cnt[2 * r];
        s1 += cnt[2 * r + 1];
    }
    part[0][t] = s0;
    part[1][t] = s1;
    __syncthreads();
    // inclusive scan of the 1024 thread sums (Hillis-Steele)
    for (int o = 1; o < 1024; o <<= 1) {
        const int a0 = t >= o ? part[0][t - o] : 0, a1 = t >= o ? part[1][t - o] : 0;
        __syncthreads();
        part[0][t] += a0;
        part[1][t] += a1;
        __syncthreads();
    }
    int e0 = part[0][t] - s0, e1 = part[1][t] - s1;
    for (int r = r0; r < r1; ++r) {
        const int n0 = cnt[2 * r], n1 = cnt[2 * r + 1];
        cnt[2 * r] = e0;
        cnt[2 * r + 1] = e1;
        e0 += n0;
        e1 += n1;
    }
    if (t == 1023) {
        tot[0] = part[0][1023];
        tot[1] = part[1][1023];
    }
}

// One wave per row: the row's band voxels of colour c go to list[c] from
// the row's offset, in increasing i.
__global__ __launch_bounds__(NT) void band_fill_kernel(uint32_t *list0, uint32_t *list1,
                                                       const int *off, const uint8_t *B, Dim d)
{
    const int lane = int(threadIdx.x) & 63;
    const int row = int(blockIdx.x) * (NT / 64) + int(threadIdx.x) / 64;
    if (row >= d.ny * d.nz) return;  // whole waves
    const int j = row % d.ny, k = row / d.ny;
    const size_t base = size_t(d.P) * row;
    int o0 = off[2 * row], o1 = off[2 * row + 1];
    const unsigned b0 = unsigned(j + k) & 1u;
    const unsigned long long below = (1ull << lane) - 1ull;
    for (int x0 = 0; x0 < d.P; x0 += 64) {
        const int t = x0 + lane;
        const bool on0 = t < d.P && B[base + t], on1 = t < d.P && B[d.half() + base + t];
        const unsigned long long m0 = __ballot(on0), m1 = __ballot(on1);
        if (on0) list0[o0 + __popcll(m0 & below)] = 2u * unsigned(base + t) + b0;
        if (on1) list1[o1 + __popcll(m1 & below)] = 2u * unsigned(base + t) + (b0 ^ 1u);
        o0 += __popcll(m0);
        o1 += __popcll(m1);
    }
}

// ---- smoothing, residual, transfers --------------------------------------

// f + hx (v-x + v+x) + hy (...) + hz (...), the sum of gauss_seidel_mex.c.
template <typename T>
__device__ __forceinline__ T gs_sum(T f, T xm, T xp, T ym, T yp, T zm, T zp, const Lap &c)
{
    return f + ((T(c.hx) * (xm + xp) + T(c.hy) * (ym + yp)) + T(c.hz) * (zm + zp));
}

// hh v + hx (v-x + v+x) + hy (...) + hz (...): Lap_h v with hh = -2 (hx + hy
// + hz) (lapmg_mex.c).
template <typename T>
__device__ __forceinline__ T lap_sum(T v, T xm, T xp, T ym, T yp, T zm, T zp, const Lap &c)
{
    const T hh = T(-2.0 * (c.hx + c.hy + c.hz));
    return ((hh * v + T(c.hx) * (xm + xp)) + T(c.hy) * (ym + yp)) + T(c.hz) * (zm + zp);
}

// One colour of a red-black Gauss-Seidel sweep (gauss_seidel_mex.c):
// v = (f + hx (v-x + v+x) + hy (...) + hz (...)) / (2 (hx + hy + hz)) on the
// voxels of M of that colour, four positions per lane.
template <typename T>
__global__ __launch_bounds__(NT) void gs_kernel(T *v, const T *f, const uint8_t *M, Dim d, Lap c,
                                                int colour)
{
    int c0, j, k, b;
    size_t p;
    if (!group4(d, c0, j, k, p, b)) return;
    b ^= colour;  // the grid has one colour: group4's parity is colour 0's
    const size_t H = d.half();
    const uint32_t m = ldm4(M + colour * H + p);
    if (m == 0) return;  // no face or position past a row's end beyond this
    T *vc = v + colour * H + p;
    Nb4<T> n;
    nb4(v + (colour ^ 1) * H, p, b, d, n);
    const V4<T> fv = ld4(f + colour * H + p);
    const T hh = T(1.0 / (2.0 * (c.hx + c.hy + c.hz)));
    V4<T> r;
#pragma unroll
    for (int e = 0; e < 4; ++e)
        r.a[e] = hh * gs_sum(fv.a[e], n.xm.a[e], n.xp.a[e], n.ym.a[e], n.yp.a[e], n.zm.a[e],
                             n.zp.a[e], c);
    if (m == 0x01010101u) {
        st4(vc, r);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (m >> (8 * e) & 1) vc[e] = r.a[e];
    }
}

// gs_kernel on the n voxels of one colour listed in idx (the band's): the
// same update, one lane per listed voxel.
template <typename T>
__global__ __launch_bounds__(NT) void gs_list_kernel(T *v, const T *f, const uint32_t *idx, int n,
                                                     Dim d, Lap c, int colour)
{
    const int t = int(blockIdx.x) * NT + int(threadIdx.x);
    if (t >= n) return;
    const uint32_t e = idx[t];
    const size_t p = e >> 1, H = d.half(), sy = size_t(d.P), sz = size_t(d.P) * d.ny;
    const T *x = v + (colour ^ 1) * H + p - 1 + (e & 1u), *o = v + (colour ^ 1) * H + p;
    const T hh = T(1.0 / (2.0 * (c.hx + c.hy + c.hz)));
    v[colour * H + p] = hh * gs_sum(f[colour * H + p], x[0], x[1], o[-ptrdiff_t(sy)], o[sy],
                                    o[-ptrdiff_t(sz)], o[sz], c);
}

// Lap_h v at the active positions m of four (zero at the others).
template <typename T>
__device__ __forceinline__ V4<T> lap4(const T *v, size_t p, int colour, int b, uint32_t m, Dim d,
                                      const Lap &c, V4<T> &vc)
{
    const size_t H = d.half();
    V4<T> r{};
    vc = ld4(v + colour * H + p);
    if (m == 0) return r;
    Nb4<T> n;
    nb4(v + (colour ^ 1) * H, p, b, d, n);
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (m >> (8 * e) & 1)
            r.a[e] = lap_sum(vc.a[e], n.xm.a[e], n.xp.a[e], n.ym.a[e], n.yp.a[e], n.zm.a[e],
                             n.zp.a[e], c);
    return r;
}

// Residual and restriction in one pass: r = f + Lap_h v on the fine mask G
// (residual_mex.c), full weighting (restrict_mex.c: 1 2 1 / 2 4 2 / 1 2 1 per
// plane, x2 in the middle plane, / 64) around the fine (2 i2 - 1, ...), onto
// G2; v2 = 0.  A block takes RX x RY x RZ coarse voxels: the residuals of the
// fine box below them go to LDS, four positions at a time and without a
// barrier in between, then each thread sums its coarse voxels' 27 in the
// order of restrict_mex.c.  r itself never reaches memory: the separate passes
// moved 200 MB and took 71 us at 258x258x178 FP32, this one takes 38 us.  (A
// block that walked the fine planes one by one, a barrier each, took 74 us:
// latency.)
constexpr int RX = 32, RY = 4, RZ = 4;
constexpr int RFY = 2 * RY + 1, RFZ = 2 * RZ + 1;
constexpr int RG = RX / 4 + 1;  // groups of four per row and colour (the last: one column)

dim3 grid_restrict(Dim d2)
{
    return dim3((d2.nx - 2 + RX - 1) / RX, (d2.ny - 2 + RY - 1) / RY, (d2.nz - 2 + RZ - 1) / RZ);
}

template <typename T>
__global__ __launch_bounds__(NT) void restrict_kernel(T *f2, T *v2, const T *f, const T *v,
                                                      const uint8_t *G, const uint8_t *G2, Dim d2,
                                                      Dim d, Lap c)
{
    __shared__ T r[RFZ][RFY][2 * RX + 2];
    int bx, by, bz;
    xcd_block3(bx, by, bz);
    const int i20 = 1 + bx * RX, j20 = 1 + by * RY, k20 = 1 + bz * RZ;  // first coarse voxel
    // the fine box starts at (2 i20 - 2, ...): position RX bx of its rows
    const size_t H = d.half();
    for (int q = int(threadIdx.x); q < RFZ * RFY * 2 * RG; q += NT) {
        const int g = q % RG, col = q / RG % 2, y = q / (2 * RG) % RFY, z = q / (2 * RG * RFY);
        const int t = RX * bx + 4 * g, j = 2 * j20 - 2 + y, k = 2 * k20 - 2 + z;
        const int b = (col + j + k) & 1;
        V4<T> o{};
        if (t < d.P && j < d.ny && k < d.nz) {
            const size_t p = size_t(t) + size_t(d.P) * (size_t(j) + size_t(d.ny) * k);
            const uint32_t m = ldm4(G + col * H + p);
            if (m != 0) {
                V4<T> vc;
                o = lap4(v, p, col, b, m, d, c, vc);
                const V4<T> fv = ld4(f + col * H + p);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    o.a[e] = (m >> (8 * e) & 1) ? fv.a[e] + o.a[e] : T(0);
            }
        }
        T *row = &r[z][y][8 * g + b];
        if (g < RG - 1) {
#pragma unroll
            for (int e = 0; e < 4; ++e) row[2 * e] = o.a[e];
        } else if (b == 0) {
            row[0] = o.a[0];
        }
    }
    __syncthreads();
    for (int q = int(threadIdx.x); q < RX * RY * RZ; q += NT) {
        const int x = q % RX, y = q / RX % RY, z = q / (RX * RY);
        const int i2 = i20 + x, j2 = j20 + y, k2 = k20 + z;
        if (!interior(d2, i2, j2, k2)) continue;
        double s = 0.0;
#pragma unroll
        for (int dk = 0; dk < 3; ++dk)
#pragma unroll
            for (int dj = 0; dj < 3; ++dj)
#pragma unroll
                for (int di = 0; di < 3; ++di)
                    s += double((di == 1 ? 2 : 1) * (dj == 1 ? 2 : 1) * (dk == 1 ? 2 : 1)) *
                         double(r[2 * z + dk][2 * y + dj][2 * x + di]);
        const size_t l2 = d2.at(i2, j2, k2);
        v2[l2] = T(0);
        f2[l2] = G2[l2] ? T(s / 64.0) : T(0);
    }
}

// correct_mex.c: v += trilinear interpolation of v2 on G (each coarse voxel
// serves the 2x2x2 fine block at (2 i2 - 1, ...)): the mean of the coarse
// values at the corners the fine voxel lies between (1, 2, 4 or 8 of them).
// Four positions per lane: they share j, k and the parity of i, so the lanes
// of a row take the same corners, and a corner row of coarse values is two
// wide loads (40 -> 31 us at 258x258x178 FP32).  Where the mask is clear the
// coarse values may lie past the row's end (v2 is allocated four positions longer).
template <typename T>
__global__ __launch_bounds__(NT) void correct_kernel(T *v, const T *v2, const uint8_t *G, Dim d,
                                                     Dim d2)
{
    int c, j, k, b;
    size_t p;
    if (!group4(d, c, j, k, p, b)) return;
    const size_t q = c * d.half() + p;
    const uint32_t m = ldm4(G + q);
    if (m == 0) return;
    const int t = int(p - size_t(d.P) * (size_t(j) + size_t(d.ny) * k));
    const int di = 1 - b, dj = (j - 1) & 1, dk = (k - 1) & 1;
    const int i2 = t + b, j2 = (j + 1 - dj) / 2, k2 = (k + 1 - dk) / 2;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    for (int ek = 0; ek <= dk; ++ek)
        for (int ej = 0; ej <= dj; ++ej) {
            // i2, i2 + 2, i2 + 4 of one colour and i2 + 1, i2 + 3 of the other
            const int ca = (i2 + j2 + ej + k2 + ek) & 1;
            const size_t row = size_t(d2.P) * (size_t(j2 + ej) + size_t(d2.ny) * (k2 + ek));
            const T *wa = v2 + size_t(ca) * d2.half() + row + (i2 >> 1);
            const T *wb = v2 + size_t(ca ^ 1) * d2.half() + row + ((i2 + 1) >> 1);
            const double w[5] = {double(wa[0]), double(wb[0]), double(wa[1]), double(wb[1]),
                                 double(wa[2])};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                s[e] += w[e];
                if (di) s[e] += w[e + 1];
            }
        }
    const double cnt = double((1 + di) * (1 + dj) * (1 + dk));
    V4<T> o = ld4(v + q);
#pragma unroll
    for (int e = 0; e < 4; ++e) o.a[e] = o.a[e] + T(s[e] / cnt);
    if (m == 0x01010101u) {
        st4(v + q, o);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (m >> (8 * e) & 1) v[q + e] = o.a[e];
    }
}

// Coarsest level, Chebyshev iteration on hh A (A = -Lap_h, hh = 1 /
// (2 (hx + hy + hz)), spectrum in [lmin, lmax]; Saad, Iterative Methods for
// Sparse Linear Systems, 2nd ed., Algorithm 12.1).  Start: r = f - A v on
// the active voxels, d = s0 hh r with s0 = 1 / theta; dz (may be null) = 0.
template <typename T>
__global__ __launch_bounds__(NT) void cheb_start_kernel(T *r, T *dn, T *dz, const T *v, const T *f,
                                                        const uint8_t *G, Dim d, Lap c, T s0)
{
    int col, j, k, b;
    size_t p;
    if (!group4(d, col, j, k, p, b)) return;
    const size_t q = col * d.half() + p;
    const uint32_t m = ldm4(G + q);
    V4<T> vc;
    V4<T> o = lap4(v, p, col, b, m, d, c, vc);
    const V4<T> fv = ld4(f + q);
    V4<T> dv;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        o.a[e] = (m >> (8 * e) & 1) ? fv.a[e] + o.a[e] : T(0);
        dv.a[e] = s0 * T(1.0 / (2.0 * (c.hx + c.hy + c.hz))) * o.a[e];
    }
    st4(r + q, o);
    st4(dn + q, dv);
    if (dz) st4(dz + q, V4<T>{});
}

// Steps of the iteration: v += d; r -= A d; d = c1 d + c2 hh r (active
// voxels; d = 0 elsewhere).
//
// Small levels, up to CS steps per launch: a block owns a CB^3 box and works
// on it and a rim of CS voxels, on which it holds r in registers and d in
// LDS, two slots; each step needs its predecessor one voxel further out, so
// what is right shrinks by a voxel per step, down to the box.  d and r go to
// other buffers than they come from (neighbour blocks read the rim); v is
// needed in the box alone.  On these levels a launch of one step takes about
// 3 us whatever the size, launch and memory latency; one of four steps takes
// 6.8 us at 34x34x24 FP32, 8.6 us at 43x50x33 FP64.
constexpr int CS = 4, CB = 8, CR = CB + 2 * CS;
constexpr int CHEB_NT = CR * CR * CR / 4;

dim3 cheb_grid(Dim d)
{
    return dim3((d.nx - 2 + CB - 1) / CB, (d.ny - 2 + CB - 1) / CB, (d.nz - 2 + CB - 1) / CB);
}

// Whether a level takes boxes.  The chip's 256 CUs hold two each (32 KB of LDS
// in FP32, 64 KB in FP64), 512 at once; more need a second round and lose.  In
// FP64 two on a CU take twice as long as one, so the time of boxes doubles at
// 257 and then stands, while that of a step per launch grows with the level:
// they meet again at about 380.  Solves of one level, one PCG iteration, boxes
// against one step per launch, MI355X: FP32 0.64 / 0.71 ms at 512 boxes
// (64x64x64), 0.79 / 0.72 at 576 (66x64x64), 2.76 / 1.46 at 4096 (256x256x30);
// FP64 0.51 / 0.58 ms at 256 (64x64x32), 0.68 / 0.59 at 288 (64x72x32), 0.72 /
// 0.68 at 360 (72x64x40), 0.78 / 0.81 at 384 (64x64x48), 0.91 / 0.95 at 512,
// 1.14 / 0.95 at 576, 4.59 / 2.75 at 4096.
template <typename T>
bool cheb_boxed(Dim d)
{
    const dim3 g = cheb_grid(d);
    const size_t n = size_t(g.x) * g.y * g.z;
    return n <= 512 && (sizeof(T) == 4 || n <= 256 || n >= 384);
}

struct ChebSteps {
    double c1[CS], c2[CS];
    int n;
};

template <typename T>
__global__ __launch_bounds__(CHEB_NT)
void cheb_steps_kernel(T *v, T *rn, T *dn, const T *r, const T *dd, const uint8_t *G, Dim d, Lap c,
                       ChebSteps cs)
{
    static_assert(CB % 4 == 0 && CS == 4, "a thread's four planes are all box or all rim");
    __shared__ T sd[2][CR][CR][CR];
    const int x = int(threadIdx.x) % CR, y = int(threadIdx.x) / CR % CR;
    const int z0 = int(threadIdx.x) / (CR * CR) * 4;  // four planes per thread
    const int i = int(blockIdx.x) * CB + 1 - CS + x, j = int(blockIdx.y) * CB + 1 - CS + y;
    const int k0 = int(blockIdx.z) * CB + 1 - CS + z0;
    const bool box = x >= CS && x < CS + CB && y >= CS && y < CS + CB && z0 >= CS && z0 < CS + CB;
    T rl[4], dl[4], vl[4];
    size_t q[4];
    uint8_t on[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        // loads do not wait for the mask; outside the grid they read voxel 0
        const bool in = interior(d, i, j, k0 + e);
        q[e] = in ? d.at(i, j, k0 + e) : 0;
        on[e] = in ? G[q[e]] : 0;
        rl[e] = r[q[e]];
        dl[e] = dd[q[e]];
        vl[e] = box ? v[q[e]] : T(0);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        dl[e] = on[e] ? dl[e] : T(0);
        sd[0][z0 + e][y][x] = dl[e];
    }
    for (int n = 0; n < cs.n; ++n) {
        const int s = n & 1;
        const T c1 = T(cs.c1[n]), c2 = T(cs.c2[n]);
        __syncthreads();
        // cells within n of the region's edge are no longer needed
        const bool need = x > n && x < CR - 1 - n && y > n && y < CR - 1 - n && z0 + 3 > n &&
                          z0 < CR - 1 - n;
        if (need) {
            T xm[4], xp[4], ym[4], yp[4], zm = z0 > 0 ? sd[s][z0 - 1][y][x] : T(0);
            const T zlast = z0 + 4 < CR ? sd[s][z0 + 4][y][x] : T(0);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                xm[e] = sd[s][z0 + e][y][x - 1];
                xp[e] = sd[s][z0 + e][y][x + 1];
                ym[e] = sd[s][z0 + e][y - 1][x];
                yp[e] = sd[s][z0 + e][y + 1][x];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                // no branch on the mask: an inactive voxel's d stays zero and
                // its r and v are not used
                const T dc = dl[e], zp = e < 3 ? dl[e < 3 ? e + 1 : 3] : zlast;
                const T ad = -lap_sum(dc, xm[e], xp[e], ym[e], yp[e], zm, zp, c);
                vl[e] = vl[e] + dc;
                rl[e] = rl[e] - ad;
                const T out = c1 * dc + c2 * T(1.0 / (2.0 * (c.hx + c.hy + c.hz))) * rl[e];
                zm = dc;
                dl[e] = on[e] ? out : T(0);
            }
        }
        if (n + 1 < cs.n) {
#pragma unroll
            for (int e = 0; e < 4; ++e) sd[s ^ 1][z0 + e][y][x] = dl[e];
        }
    }
    if (box) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (on[e]) {
                v[q[e]] = vl[e];
                rn[q[e]] = rl[e];
                dn[q[e]] = dl[e];
            }
    }
}

// Large levels, one step per launch, four positions per lane: every field
// passes through memory once a step, where a box with its rim loads and
// updates 8 voxels for each of its own.  r is updated in place, d goes to
// another buffer (its neighbours are read), zero at inactive voxels already.
template <typename T>
__global__ __launch_bounds__(NT) void cheb_step_kernel(T *v, T *r, T *dn, const T *dd,
                                                       const uint8_t *G, Dim d, Lap c, T c1, T c2)
{
    int col, j, k, b;
    size_t p;
    if (!group4(d, col, j, k, p, b)) return;
    const size_t q = col * d.half() + p;
    const uint32_t m = ldm4(G + q);
    if (m == 0) return;
    V4<T> dc;
    const V4<T> la = lap4(dd, p, col, b, m, d, c, dc);
    V4<T> vv = ld4(v + q), rv = ld4(r + q), o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        // d, r and their Laplacian are zero at an inactive voxel
        vv.a[e] = vv.a[e] + dc.a[e];
        rv.a[e] = rv.a[e] + la.a[e];
        o.a[e] = c1 * dc.a[e] + c2 * T(1.0 / (2.0 * (c.hx + c.hy + c.hz))) * rv.a[e];
    }
    st4(v + q, vv);
    st4(r + q, rv);
    st4(dn + q, o);
}

// ---- PCG vector kernels ----------------------------------------------------

template <typename T>
__global__ __launch_bounds__(NT) void zero_kernel(T *a, size_t n)
{
    const size_t l = size_t(blockIdx.x) * NT + threadIdx.x;
    if (l < n) a[l] = T(0);
}

// r -= q
template <typename T>
__global__ __launch_bounds__(NT) void sub_kernel(T *r, const T *q, size_t n)
{
    const size_t l = size_t(blockIdx.x) * NT + threadIdx.x;
    if (l < n) r[l] = r[l] - q[l];
}

// The block's sum of acc in a fixed order, to part[block].
__device__ __forceinline__ void block_part(double acc, double *part, int block)
{
    __shared__ double red[NT];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = NT / 2; s > 0; s >>= 1) {
        if (int(threadIdx.x) < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[block] = red[0];
}

// partial sums of a[l] * b[l] over a fixed grid of DOT_BLOCKS blocks (each
// thread strides the array, four positions at a time; fixed order, so the
// result is reproducible)
template <typename T>
__global__ __launch_bounds__(NT) void dot_kernel(const T *a, const T *b, size_t n, double *part)
{
    double acc = 0.0;
    for (size_t l = 4 * (size_t(blockIdx.x) * NT + threadIdx.x); l < n;
         l += 4 * size_t(DOT_BLOCKS) * NT) {
        const V4<T> x = ld4(a + l), y = ld4(b + l);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc += double(x.a[e]) * double(y.a[e]);
    }
    block_part(acc, part, int(blockIdx.x));
}

// RES = false: q = A p (A = -Lap_h, lapmg_mex.c) on G, 0 elsewhere, and the
// partial sums of p . q.  RES = true: the partial sums of r . r, r = q - A p
// on G, 0 elsewhere (residual_mex.c), and nothing written.  A block takes one
// contiguous range of positions, both colours of it (each is the other's
// neighbours), and the blocks of an XCD contiguous ranges: a slab of planes.
template <typename T, bool RES>
__global__ __launch_bounds__(NT) void apply_kernel(T *q, const T *p, const uint8_t *G, Dim d,
                                                   Lap c, double *part)
{
    const int blk = xcd_block();
    const size_t H = d.half(), ng = H / 4, per = (ng + DOT_BLOCKS - 1) / DOT_BLOCKS;
    const size_t g0 = per * blk, g1 = min(ng, g0 + per);
    const unsigned g4 = unsigned(d.P) / 4;
    double acc = 0.0;
    for (size_t g = g0 + threadIdx.x; g < g1; g += NT) {
        const unsigned row = unsigned(g / g4);
        const int par = int(row % unsigned(d.ny) + row / unsigned(d.ny)) & 1;
#pragma unroll
        for (int col = 0; col < 2; ++col) {
            const size_t l = 4 * g;
            const uint32_t m = ldm4(G + col * H + l);
            V4<T> pc;
            V4<T> o = lap4(p, l, col, par ^ col, m, d, c, pc);
            if (RES) {
                const V4<T> f = ld4(q + col * H + l);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    o.a[e] = (m >> (8 * e) & 1) ? f.a[e] + o.a[e] : T(0);
                    acc += double(o.a[e]) * double(o.a[e]);
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    o.a[e] = (m >> (8 * e) & 1) ? -o.a[e] : T(0);
                    acc += double(pc.a[e]) * double(o.a[e]);
                }
                st4(q + col * H + l, o);
            }
        }
    }
    block_part(acc, part, blk);
}

__global__ __launch_bounds__(NT) void sum_kernel(const double *part, int nb, double *out)
{
    __shared__ double red[NT];
    double s = 0.0;
    for (int b = threadIdx.x; b < nb; b += NT) s += part[b];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int k = NT / 2; k > 0; k >>= 1) {
        if (int(threadIdx.x) < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = red[0];
}

// The PCG loop's scalars on the device (mgpcg_mex.c: mx_pcg), so that an
// iteration reads back only ||r||^2 and the breakdown flag.
struct Pcg {
    double rho, prevrho, pq, rr;
    int brk;  // rho or pq not positive: the reference's loop breaks there
    int pad;
};

// sum_kernel's reduction into the PCG scalars.  WHAT 0: rr; 1: rho, the
// previous rho kept as prevrho, breakdown when !(rho > 0); 2: pq,
// breakdown when !(pq > 0).
template <int WHAT>
__global__ __launch_bounds__(NT) void pcg_sum_kernel(const double *part, int nb, Pcg *g)
{
    __shared__ double red[NT];
    double s = 0.0;
    for (int b = threadIdx.x; b < nb; b += NT) s += part[b];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int k = NT / 2; k > 0; k >>= 1) {
        if (int(threadIdx.x) < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x != 0) return;
    const double v = red[0];
    if (WHAT == 0) {
        g->rr = v;
    } else if (WHAT == 1) {
        g->prevrho = g->rho;
        g->rho = v;
        if (!(v > 0.0)) g->brk = 1;
    } else {
        g->pq = v;
        if (!(v > 0.0)) g->brk = 1;
    }
}

// p = q + beta p with beta = rho / prevrho (skipped after a breakdown)
template <typename T>
__global__ __launch_bounds__(NT) void xpby_pcg_kernel(T *p, const T *q, const Pcg *g, size_t n)
{
    if (g->brk) return;
    const T beta = T(g->rho / g->prevrho);
    const size_t l = 4 * (size_t(blockIdx.x) * NT + threadIdx.x);
    if (l >= n) return;
    V4<T> pv = ld4(p + l);
    const V4<T> qv = ld4(q + l);
#pragma unroll
    for (int e = 0; e < 4; ++e) pv.a[e] = beta * pv.a[e] + qv.a[e];
    st4(p + l, pv);
}

// x += a p; r -= a q with a = rho / pq (skipped after a breakdown), and the
// partial sums of r . r
template <typename T>
__global__ __launch_bounds__(NT) void update_pcg_kernel(T *x, T *r, const T *p, const T *q,
                                                        const Pcg *g, size_t n, double *part)
{
    const bool brk = g->brk != 0;
    const T a = brk ? T(0) : T(g->rho / g->pq);
    double acc = 0.0;
    for (size_t l = 4 * (size_t(blockIdx.x) * NT + threadIdx.x); l < n;
         l += 4 * size_t(DOT_BLOCKS) * NT) {
        V4<T> rv = ld4(r + l);
        if (!brk) {
            V4<T> xv = ld4(x + l);
            const V4<T> pv = ld4(p + l), qv = ld4(q + l);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                xv.a[e] = xv.a[e] + a * pv.a[e];
                rv.a[e] = rv.a[e] - a * qv.a[e];
            }
            st4(x + l, xv);
            st4(r + l, rv);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) acc += double(rv.a[e]) * double(rv.a[e]);
    }
    block_part(acc, part, int(blockIdx.x));
}

unsigned g1(size_t n) { return unsigned((n + NT - 1) / NT); }
unsigned g1v(size_t n) { return unsigned((n / 4 + NT - 1) / NT); }  // four positions per lane

size_t al(size_t n) { return (n + 255) / 256 * 256; }

// ---- the solver --------------------------------------------------------------

template <typename T>
struct Level {
    Dim d;
    Lap c;
    T *v, *f;
    uint8_t *G, *B;
    uint32_t *bl;  // band voxels of colour 0 from bl, of colour 1 from bl + (nat() + 1) / 2
    int bn[2];  // their counts (host copy)
};

template <typename T>
struct Solver {
    int L;
    Level<T> lv[MAX_LEVELS];
    T *x, *p;           // PCG iterate and direction (level-0 size)
    T *cd[2], *cr[2];   // coarsest level: the Chebyshev d and r (cr[1]: where boxes update it)
    uint8_t *gn[2];     // masks of a level and the next in natural order (set-up)
    uint8_t *tmp;       // band seed scratch (level-0 size)
    int *rowcnt, *btot; // band list construction: per-row counts, totals per level
    double *part, *sum; // reductions
    Pcg *pcg;           // the PCG scalars
};

// Level sizes: the padded grid, then ((n - 2 + 1) >> 1) + 2 per level
// (mgpcg_mex.c: mx_init).
int level_dims(const size_t sz[3], int L, Dim *d)
{
    d[0] = make_dim(int(sz[0]) + 2, int(sz[1]) + 2, int(sz[2]) + 2);
    for (int i = 1; i < L; ++i)
        d[i] = make_dim(((d[i - 1].nx - 2 + 1) >> 1) + 2, ((d[i - 1].ny - 2 + 1) >> 1) + 2,
                        ((d[i - 1].nz - 2 + 1) >> 1) + 2);
    return QSM_OK;
}

template <typename T>
size_t solver_layout(const size_t sz[3], const double vsz[3], int L, Solver<T> *s, char *base)
{
    Dim d[MAX_LEVELS];
    level_dims(sz, L, d);
    size_t off = 0;
    auto take = [&](size_t b) { char *p = base ? base + off : nullptr; off += al(b); return p; };
    for (int i = 0; i < L; ++i) {
        const size_t n = d[i].n();
        char *pv = take((n + 4) * sizeof(T)), *pf = take(n * sizeof(T));
        char *pG = take(n), *pB = take(n);
        // band lists on the levels that smooth (not the coarsest)
        char *pl = i < L - 1 ? take((d[i].nat() + 1) * sizeof(uint32_t)) : nullptr;
        if (s)
            s->lv[i] = Level<T>{d[i], lap_at(vsz, i), reinterpret_cast<T *>(pv),
                                reinterpret_cast<T *>(pf), reinterpret_cast<uint8_t *>(pG),
                                reinterpret_cast<uint8_t *>(pB), reinterpret_cast<uint32_t *>(pl),
                                {0, 0}};
    }
    const size_t n0 = d[0].n();
    char *px = take(n0 * sizeof(T)), *pp = take(n0 * sizeof(T)), *pt = take(d[0].nat());
    char *pg0 = take(d[0].nat()), *pg1 = L > 1 ? take(d[1].nat()) : nullptr;
    char *prc = take(2 * size_t(d[0].ny) * d[0].nz * sizeof(int));
    char *pbt = take(2 * MAX_LEVELS * sizeof(int));
    const size_t nc = d[L - 1].n();
    char *pc[4];
    for (int a = 0; a < 4; ++a)
        pc[a] = a < 3 || cheb_boxed<T>(d[L - 1]) ? take(nc * sizeof(T)) : nullptr;
    char *ppart = take(DOT_BLOCKS * sizeof(double)), *psum = take(sizeof(double));
    char *ppcg = take(sizeof(Pcg));
    if (s) {
        s->L = L;
        s->x = reinterpret_cast<T *>(px);
        s->p = reinterpret_cast<T *>(pp);
        for (int a = 0; a < 2; ++a) {
            s->cd[a] = reinterpret_cast<T *>(pc[a]);
            s->cr[a] = reinterpret_cast<T *>(pc[2 + a]);
        }
        s->gn[0] = reinterpret_cast<uint8_t *>(pg0);
        s->gn[1] = reinterpret_cast<uint8_t *>(pg1);
        s->tmp = reinterpret_cast<uint8_t *>(pt);
        s->rowcnt = reinterpret_cast<int *>(prc);
        s->btot = reinterpret_cast<int *>(pbt);
        s->part = reinterpret_cast<double *>(ppart);
        s->sum = reinterpret_cast<double *>(psum);
        s->pcg = reinterpret_cast<Pcg *>(ppcg);
    }
    return off;
}

// The sum of the partial sums in s.part, read back.
template <typename T>
int read_sum(Solver<T> &s, double &out, hipStream_t st)
{
    sum_kernel<<<1, NT, 0, st>>>(s.part, DOT_BLOCKS, s.sum);
    QSM_HIP(hipGetLastError());
    QSM_HIP(hipMemcpyAsync(&out, s.sum, sizeof(double), hipMemcpyDeviceToHost, st));
    QSM_HIP(hipStreamSynchronize(st));
    return QSM_OK;
}

template <typename T>
int dot(const T *a, const T *b, size_t n, Solver<T> &s, double &out, hipStream_t st)
{
    dot_kernel<T><<<DOT_BLOCKS, NT, 0, st>>>(a, b, n, s.part);
    QSM_HIP(hipGetLastError());
    return read_sum(s, out, st);
}

// n red-black sweeps on mask M.  Forward sweeps take the even colour
// ((i + j + k) even) first; reverse sweeps start from the volume's far
// corner, whose colour is that of parity nx + 1 (gauss_seidel_mex.c:141-163).
template <typename T>
int smooth(Level<T> &L, const uint8_t *M, int n, bool reverse, hipStream_t st)
{
    const dim3 g = grid4(L.d, 1);
    const int first = reverse ? ((L.d.nx + 1) & 1) : 0;
    for (int s = 0; s < n; ++s)
        for (int h = 0; h < 2; ++h) {
            gs_kernel<T><<<g, NT, 0, st>>>(L.v, L.f, M, L.d, L.c, first ^ h);
            QSM_HIP(hipGetLastError());
        }
    return QSM_OK;
}

// n red-black sweeps on the level's band, from its index lists; the colour
// order of smooth().
template <typename T>
int smooth_band(Level<T> &L, int n, bool reverse, hipStream_t st)
{
    const int first = reverse ? ((L.d.nx + 1) & 1) : 0;
    const uint32_t *list[2] = {L.bl, L.bl + (L.d.nat() + 1) / 2};
    for (int s = 0; s < n; ++s)
        for (int h = 0; h < 2; ++h) {
            const int c = first ^ h;
            if (L.bn[c] == 0) continue;
            gs_list_kernel<T><<<(L.bn[c] + NT - 1) / NT, NT, 0, st>>>(L.v, L.f, list[c], L.bn[c],
                                                                     L.d, L.c, c);
            QSM_HIP(hipGetLastError());
        }
    return QSM_OK;
}

// Spectrum bounds of hh A on the level's box (interior nx-2 x ny-2 x nz-2,
// Dirichlet): lmin = hh sum_a 2 h_a (1 - cos(pi / (m_a + 1))), lmax = 2 -
// lmin; the Chebyshev degree that reduces the error by CHEB_EPS over them.
struct Cheb {
    double lmin, lmax;
    int K;
};

Cheb cheb_of(const Dim &d, const Lap &c)
{
    const double pi = 3.14159265358979323846;
    const double hh = 1.0 / (2.0 * (c.hx + c.hy + c.hz));
    const double w[3] = {c.hx, c.hy, c.hz};
    const int m[3] = {d.nx - 2, d.ny - 2, d.nz - 2};
    double lmin = 0.0;
    for (int a = 0; a < 3; ++a) lmin += hh * 2.0 * w[a] * (1.0 - std::cos(pi / (m[a] + 1)));
    const double lmax = 2.0 - lmin;
    const double sigma = (lmax + lmin) / (lmax - lmin);
    const int K = int(std::ceil(std::acosh(1.0 / CHEB_EPS) / std::acosh(sigma)));
    return Cheb{lmin, lmax, std::max(1, std::min(K, CHEB_MAX))};
}

// The coarsest level: K Chebyshev steps from the current v (restriction
// zeroed it, except on a one-level hierarchy's later cycles).
template <typename T>
int coarse_solve(Solver<T> &s, Level<T> &L, hipStream_t st)
{
    const Cheb ch = cheb_of(L.d, L.c);
    const double theta = 0.5 * (ch.lmax + ch.lmin), delta = 0.5 * (ch.lmax - ch.lmin);
    const double sigma = theta / delta;
    const bool boxed = cheb_boxed<T>(L.d);
    cheb_start_kernel<T><<<grid4(L.d, 2), NT, 0, st>>>(s.cr[0], s.cd[0], boxed ? nullptr : s.cd[1],
                                                       L.v, L.f, L.G, L.d, L.c, T(1.0 / theta));
    QSM_HIP(hipGetLastError());
    double rho = 1.0 / sigma;
    int cur = 0;
    if (!boxed) {
        for (int k = 0; k < ch.K; ++k, cur ^= 1) {
            const double rho1 = 1.0 / (2.0 * sigma - rho);
            cheb_step_kernel<T><<<grid4(L.d, 2), NT, 0, st>>>(
                L.v, s.cr[0], s.cd[cur ^ 1], s.cd[cur], L.G, L.d, L.c, T(rho1 * rho),
                T(2.0 * rho1 / delta));
            QSM_HIP(hipGetLastError());
            rho = rho1;
        }
        return QSM_OK;
    }
    const dim3 g = cheb_grid(L.d);
    for (int k = 0; k < ch.K; k += CS) {
        ChebSteps cs;
        cs.n = std::min(CS, ch.K - k);
        for (int n = 0; n < cs.n; ++n) {
            const double rho1 = 1.0 / (2.0 * sigma - rho);
            cs.c1[n] = rho1 * rho;
            cs.c2[n] = 2.0 * rho1 / delta;
            rho = rho1;
        }
        cheb_steps_kernel<T><<<g, CHEB_NT, 0, st>>>(L.v, s.cr[cur ^ 1], s.cd[cur ^ 1], s.cr[cur],
                                                    s.cd[cur], L.G, L.d, L.c, cs);
        QSM_HIP(hipGetLastError());
        cur ^= 1;
    }
    return QSM_OK;
}

struct MgParams {
    double tol;
    int cycles, mu, npre, npost, nboundary;
};

// mgpcg_mex.c: mx_cycle on level l.
template <typename T>
int cycle(Solver<T> &s, int l, const MgParams &m, hipStream_t st)
{
    int rc;
    Level<T> &L = s.lv[l];
    if (l < s.L - 1) {
        const int bs = (1 << l) * m.nboundary;
        if ((rc = smooth(L, L.G, m.npre, false, st))) return rc;
        if ((rc = smooth_band(L, bs, false, st))) return rc;
        Level<T> &C = s.lv[l + 1];
        restrict_kernel<T><<<grid_restrict(C.d), NT, 0, st>>>(C.f, C.v, L.f, L.v, L.G, C.G, C.d,
                                                              L.d, L.c);
        QSM_HIP(hipGetLastError());
        for (int i = 0; i < m.mu; ++i) {
            if ((rc = cycle(s, l + 1, m, st))) return rc;
            if (l + 1 == s.L - 1) break;
        }
        correct_kernel<T><<<grid4(L.d, 2), NT, 0, st>>>(L.v, C.v, L.G, L.d, C.d);
        QSM_HIP(hipGetLastError());
        if ((rc = smooth_band(L, bs, true, st))) return rc;
        if ((rc = smooth(L, L.G, m.npost, true, st))) return rc;
    } else {
        if ((rc = coarse_solve(s, L, st))) return rc;
    }
    return QSM_OK;
}

// Solves -Lap v = f on the mask (sz, unpadded, device), v out (sz).  src:
// f itself, or with unwrap != 0 the wrapped Laplacian d2u whose right-hand
// side is -m .* d2u (unwrapLaplacian.m:84).
//
// x0 (may be null): the initial guess (sz, device); PCG then starts from
// r = f - A x0, with the stopping rule still relative to ||f||
// (mgpcg_mex.c: mx_pcg).
template <typename T>
int mgpcg_t(const T *src, bool unwrap, const uint8_t *mask, const size_t sz[3],
            const double vsz[3], double tol, int maxit, const MgParams &m, int nlevels, T *v,
            void *work, int *iters, double *resnorm, hipStream_t st, const T *x0 = nullptr)
{
    int rc;
    Solver<T> s;
    // fields start at multiples of 256 bytes whatever the caller's pointer
    char *base = reinterpret_cast<char *>(al(reinterpret_cast<uintptr_t>(work)));
    solver_layout<T>(sz, vsz, nlevels, &s, base);
    Level<T> &L0 = s.lv[0];
    const size_t n0 = L0.d.n();
    const dim3 b(BX, BY);
    // level 0: r (held in f) = padded right-hand side; masks of the hierarchy
    // (built in natural order, kept split); v zero, which faces and inactive
    // voxels stay (restrict_kernel clears the rest for each cycle)
    pad_kernel<T><<<grid4(L0.d, 2), NT, 0, st>>>(L0.f, src, s.gn[0], mask, L0.d,
                                                 unwrap ? T(-1) : T(0));
    QSM_HIP(hipGetLastError());
    for (int l = 0; l < s.L; ++l) {
        Level<T> &L = s.lv[l];
        uint8_t *gn = s.gn[l & 1];
        if (l > 0) {
            coarsen_kernel<<<grid3(L.d), b, 0, st>>>(gn, s.gn[(l - 1) & 1], L.d, s.lv[l - 1].d);
            zero_kernel<T><<<g1(L.d.n()), NT, 0, st>>>(L.v, L.d.n());
            QSM_HIP(hipGetLastError());
        }
        band_seed_kernel<<<grid3(L.d), b, 0, st>>>(s.tmp, gn, L.d);
        band_kernel<<<grid4(L.d, 2), NT, 0, st>>>(L.B, L.G, s.tmp, gn, L.d);
        QSM_HIP(hipGetLastError());
        if (l < s.L - 1) {
            // the band's index lists per colour
            const int rows = L.d.ny * L.d.nz, rb = (rows + NT / 64 - 1) / (NT / 64);
            band_count_kernel<<<rb, NT, 0, st>>>(s.rowcnt, L.B, L.d);
            band_scan_kernel<<<1, 1024, 0, st>>>(s.rowcnt, rows, s.btot + 2 * l);
            band_fill_kernel<<<rb, NT, 0, st>>>(L.bl, L.bl + (L.d.nat() + 1) / 2, s.rowcnt, L.B,
                                                L.d);
            QSM_HIP(hipGetLastError());
        }
    }
    if (s.L > 1) {
        int tot[2 * MAX_LEVELS];
        QSM_HIP(hipMemcpyAsync(tot, s.btot, 2 * (s.L - 1) * sizeof(int), hipMemcpyDeviceToHost,
                               st));
        QSM_HIP(hipStreamSynchronize(st));
        for (int l = 0; l < s.L - 1; ++l) {
            s.lv[l].bn[0] = tot[2 * l];
            s.lv[l].bn[1] = tot[2 * l + 1];
        }
    }
    // PCG (mgpcg_mex.c: mx_pcg): reltol from ||f||, then r = f - A x0
    zero_kernel<T><<<g1(n0), NT, 0, st>>>(s.p, n0);
    QSM_HIP(hipGetLastError());
    T *r = L0.f, *q = L0.v;
    double res;
    if ((rc = dot(r, r, n0, s, res, st))) return rc;
    res = std::sqrt(res);
    const double reltol = tol * res;
    if (x0) {
        pad_kernel<T><<<grid4(L0.d, 2), NT, 0, st>>>(s.x, x0, nullptr, mask, L0.d, T(0));
        apply_kernel<T, false><<<DOT_BLOCKS, NT, 0, st>>>(q, s.x, L0.G, L0.d, L0.c, s.part);
        sub_kernel<T><<<g1(n0), NT, 0, st>>>(r, q, n0);
        QSM_HIP(hipGetLastError());
        if ((rc = dot(r, r, n0, s, res, st))) return rc;
        res = std::sqrt(res);
    } else {
        zero_kernel<T><<<g1(n0), NT, 0, st>>>(s.x, n0);
        QSM_HIP(hipGetLastError());
    }
    // rho, prevrho, pq and ||r||^2 stay on the device; each iteration reads
    // back ||r||^2 and the breakdown flag once, at its end
    const Pcg g0{1.0, 1.0, 0.0, 0.0, 0, 0};  // rho = 1 before the first iteration
    QSM_HIP(hipMemcpyAsync(s.pcg, &g0, sizeof(Pcg), hipMemcpyHostToDevice, st));
    int it = 0;
    for (; it < maxit; ++it) {
        if (res <= reltol) break;
        // q = M \ r: m.cycles V-cycles from q = 0 (mgpcg_mex.c: mx_mg; with
        // mgopts.tol > 0 they stop once ||r - A q|| < mgopts.tol ||r||)
        zero_kernel<T><<<g1(n0), NT, 0, st>>>(q, n0);
        QSM_HIP(hipGetLastError());
        const double mgtol = m.tol > 0.0 ? m.tol * res : 0.0;
        for (int k = 0; k < m.cycles; ++k) {
            if (m.tol > 0.0) {
                apply_kernel<T, true><<<DOT_BLOCKS, NT, 0, st>>>(L0.f, L0.v, L0.G, L0.d, L0.c,
                                                                 s.part);
                QSM_HIP(hipGetLastError());
                double rn;
                if ((rc = read_sum(s, rn, st))) return rc;
                if (std::sqrt(rn) < mgtol) break;
            }
            if ((rc = cycle(s, 0, m, st))) return rc;
        }
        // rho = r.q (prevrho = the last one); breakdown when !(rho > 0): the
        // residual is exactly zero on the mask (the rule above never stops
        // a right-hand side that is nonzero off the mask, since ||r|| counts
        // the whole array), so no direction is left
        dot_kernel<T><<<DOT_BLOCKS, NT, 0, st>>>(r, q, n0, s.part);
        pcg_sum_kernel<1><<<1, NT, 0, st>>>(s.part, DOT_BLOCKS, s.pcg);
        // p = q + (rho / prevrho) p; q = A p; pq = p.q (breakdown: !(pq > 0))
        xpby_pcg_kernel<T><<<g1v(n0), NT, 0, st>>>(s.p, q, s.pcg, n0);
        apply_kernel<T, false><<<DOT_BLOCKS, NT, 0, st>>>(q, s.p, L0.G, L0.d, L0.c, s.part);
        pcg_sum_kernel<2><<<1, NT, 0, st>>>(s.part, DOT_BLOCKS, s.pcg);
        // x += (rho / pq) p; r -= (rho / pq) q; ||r||^2
        update_pcg_kernel<T><<<DOT_BLOCKS, NT, 0, st>>>(s.x, r, s.p, q, s.pcg, n0, s.part);
        pcg_sum_kernel<0><<<1, NT, 0, st>>>(s.part, DOT_BLOCKS, s.pcg);
        QSM_HIP(hipGetLastError());
        Pcg g;
        QSM_HIP(hipMemcpyAsync(&g, s.pcg, sizeof(Pcg), hipMemcpyDeviceToHost, st));
        QSM_HIP(hipStreamSynchronize(st));
        if (g.brk) break;  // x and r are as the reference leaves them
        res = std::sqrt(g.rr);
        if (resnorm) resnorm[it] = res;
    }
    if (iters) *iters = it;
    unpad_kernel<T><<<grid3(L0.d), b, 0, st>>>(v, s.x, L0.d);
    QSM_HIP(hipGetLastError());
    return QSM_OK;
}

int default_levels(const size_t sz[3])
{
    // mgpcg.m:51: max(1, floor(log2(min(size(f)))) - 3)
    const size_t mn = std::min(sz[0], std::min(sz[1], sz[2]));
    return std::max(1, int(std::floor(std::log2(double(mn)))) - 3);
}

int check_mg(int dtype, const size_t sz[3], const double vsz[3], const qsm_mg_opts *o, int &L)
{
    QSM_ARG(dtype == QSM_F64 || dtype == QSM_F32, "bad dtype");
    QSM_ARG(sz && vsz && o, "null pointer");
    int rc = check_grid(sz, vsz, 1);
    if (rc) return rc;
    L = o->nlevels > 0 ? o->nlevels : default_levels(sz);
    QSM_ARG(L >= 1 && L <= MAX_LEVELS, "mgopts.nlevels %d out of range 1..%d", L, MAX_LEVELS);
    Dim d[MAX_LEVELS];
    level_dims(sz, L, d);
    QSM_ARG(d[L - 1].nx > 2 && d[L - 1].ny > 2 && d[L - 1].nz > 2,
            "mgopts.nlevels %d too many for this size", L);
    QSM_ARG(o->maxit >= 1 && o->mu >= 1 && o->npre >= 0 && o->npost >= 0 && o->nboundary >= 0 &&
            std::isfinite(o->tol), "invalid mgopts");
    return QSM_OK;
}

}  // namespace

extern "C" {

void qsm_mg_opts_default(qsm_mg_opts *o)
{
    // mgpcg.m:11-52
    o->tol = -1.0;
    o->maxit = 1;
    o->mu = 1;
    o->npre = 1;
    o->npost = 1;
    o->nboundary = 2;
    o->nlevels = 0;
}

size_t qsm_mgpcg_work_bytes(int dtype, const size_t sz[3], int nlevels)
{
    if (!sz) return 0;
    const int L = nlevels > 0 ? nlevels : default_levels(sz);
    if (L < 1 || L > MAX_LEVELS) return 0;
    const double one[3] = {1.0, 1.0, 1.0};
    // 255 more: the work space may start anywhere
    return 255 + (dtype == QSM_F32 ? solver_layout<float>(sz, one, L, nullptr, nullptr)
                                   : solver_layout<double>(sz, one, L, nullptr, nullptr));
}

int qsm_mgpcg_dev(int dtype, const void *f, const uint8_t *mask, const size_t sz[3],
                  const double vsz[3], double tol, int maxit, const qsm_mg_opts *mgopts, void *v,
                  void *work, int *iters, double *resnorm, void *stream)
{
    int L, rc = check_mg(dtype, sz, vsz, mgopts, L);
    if (rc) return rc;
    QSM_ARG(f && mask && v && work, "null pointer");
    QSM_ARG(maxit >= 1 && std::isfinite(tol), "tol must be finite and maxit >= 1");
    const MgParams m{mgopts->tol, mgopts->maxit, mgopts->mu, mgopts->npre, mgopts->npost,
                     mgopts->nboundary};
    const hipStream_t st = as_stream(stream);
    return dtype == QSM_F64
        ? mgpcg_t<double>(static_cast<const double *>(f), false, mask, sz, vsz, tol, maxit, m, L,
                          static_cast<double *>(v), work, iters, resnorm, st)
        : mgpcg_t<float>(static_cast<const float *>(f), false, mask, sz, vsz, tol, maxit, m, L,
                         static_cast<float *>(v), work, iters, resnorm, st);
}

int qsm_mgpcg(int dtype, const void *f, const uint8_t *mask, const size_t sz[3],
              const double vsz[3], double tol, int maxit, const qsm_mg_opts *mgopts, void *v,
              int *iters, double *resnorm)
{
    int L, rc = check_mg(dtype, sz, vsz, mgopts, L);
    if (rc) return rc;
    QSM_ARG(f && mask && v, "null pointer");
    QSM_ARG(maxit >= 1 && std::isfinite(tol), "tol must be finite and maxit >= 1");
    if ((rc = ensure_device())) return rc;
    const size_t N = sz[0] * sz[1] * sz[2], es = dtype_size(dtype);
    DevBuf df, dm, dv, dw;
    if ((rc = df.alloc(N * es)) || (rc = dm.alloc(N)) || (rc = dv.alloc(N * es))
        || (rc = dw.alloc(qsm_mgpcg_work_bytes(dtype, sz, L))))
        return rc;
    QSM_HIP(hipMemcpy(df.p, f, N * es, hipMemcpyHostToDevice));
    QSM_HIP(hipMemcpy(dm.p, mask, N, hipMemcpyHostToDevice));
    if ((rc = qsm_mgpcg_dev(dtype, df.p, static_cast<const uint8_t *>(dm.p), sz, vsz, tol, maxit,
                            mgopts, dv.p, dw.p, iters, resnorm, nullptr)))
        return rc;
    QSM_HIP(hipStreamSynchronize(nullptr));
    QSM_HIP(hipMemcpy(v, dv.p, N * es, hipMemcpyDeviceToHost));
    return QSM_OK;
}

int qsm_mgpcg_x0(int dtype, const void *f, const uint8_t *mask, const size_t sz[3],
                 const double vsz[3], double tol, int maxit, const qsm_mg_opts *mgopts, void *v,
                 int *iters, double *resnorm)
{
    int L, rc = check_mg(dtype, sz, vsz, mgopts, L);
    if (rc) return rc;
    QSM_ARG(f && mask && v, "null pointer");
    QSM_ARG(maxit >= 0 && std::isfinite(tol), "tol must be finite and maxit >= 0");
    if ((rc = ensure_device())) return rc;
    const size_t N = sz[0] * sz[1] * sz[2], es = dtype_size(dtype);
    DevBuf df, dm, dv, dx, dw;
    if ((rc = df.alloc(N * es)) || (rc = dm.alloc(N)) || (rc = dv.alloc(N * es))
        || (rc = dx.alloc(N * es)) || (rc = dw.alloc(qsm_mgpcg_work_bytes(dtype, sz, L))))
        return rc;
    QSM_HIP(hipMemcpy(df.p, f, N * es, hipMemcpyHostToDevice));
    QSM_HIP(hipMemcpy(dm.p, mask, N, hipMemcpyHostToDevice));
    QSM_HIP(hipMemcpy(dx.p, v, N * es, hipMemcpyHostToDevice));
    const MgParams m{mgopts->tol, mgopts->maxit, mgopts->mu, mgopts->npre, mgopts->npost,
                     mgopts->nboundary};
    const hipStream_t st = nullptr;
    rc = dtype == QSM_F64
        ? mgpcg_t<double>(static_cast<const double *>(df.p), false,
                          static_cast<const uint8_t *>(dm.p), sz, vsz, tol, maxit, m, L,
                          static_cast<double *>(dv.p), dw.p, iters, resnorm, st,
                          static_cast<const double *>(dx.p))
        : mgpcg_t<float>(static_cast<const float *>(df.p), false,
                         static_cast<const uint8_t *>(dm.p), sz, vsz, tol, maxit, m, L,
                         static_cast<float *>(dv.p), dw.p, iters, resnorm, st,
                         static_cast<const float *>(dx.p));
    if (rc) return rc;
    QSM_HIP(hipStreamSynchronize(nullptr));
    QSM_HIP(hipMemcpy(v, dv.p, N * es, hipMemcpyDeviceToHost));
    return QSM_OK;
}

int qsm_unwrap_laplacian_dev(int dtype, const void *u, const uint8_t *mask, const size_t sz[3],
                             const double vsz[3], void *uphas, void *d2u, void *work,
                             int *iters, void *stream)
{
    // unwrapLaplacian.m:78-98 on an already cropped volume: d2u = lapw(u,
    // h), then mgpcg(-m .* d2u, m, h, 1e-8, ceil(sqrt(numel(m))), mgopts
    // with maxit = npre = npost = nboundary = 2)
    qsm_mg_opts o;
    qsm_mg_opts_default(&o);
    o.maxit = 2;
    o.npre = 2;
    o.npost = 2;
    o.nboundary = 2;
    int L, rc = check_mg(dtype, sz, vsz, &o, L);
    if (rc) return rc;
    QSM_ARG(u && mask && uphas && d2u && work, "null pointer");
    const size_t N = sz[0] * sz[1] * sz[2];
    const hipStream_t st = as_stream(stream);
    // lapw leaves the faces untouched: they are zero in the reference
    QSM_HIP(hipMemsetAsync(d2u, 0, N * dtype_size(dtype), st));
    if ((rc = qsm_lapw_dev(dtype, d2u, u, sz, vsz, stream))) return rc;
    const int maxit = int(std::ceil(std::sqrt(double(N))));
    const MgParams m{o.tol, o.maxit, o.mu, o.npre, o.npost, o.nboundary};
    return dtype == QSM_F64
        ? mgpcg_t<double>(static_cast<const double *>(d2u), true, mask, sz, vsz, 1e-8, maxit, m,
                          L, static_cast<double *>(uphas), work, iters, nullptr, st)
        : mgpcg_t<float>(static_cast<const float *>(d2u), true, mask, sz, vsz, 1e-8, maxit, m, L,
                         static_cast<float *>(uphas), work, iters, nullptr, st);
}

int qsm_unwrap_laplacian(int dtype, const void *phas, const uint8_t *mask, const size_t sz[3],
                         size_t nechoes, const double vsz[3], void *uphas, void *d2phas)
{
    // unwrapLaplacian.m:60-75: crop to the mask's box grown by one voxel
    // (clamped to the volume), per echo unwrap_, uncrop into zeros
    QSM_ARG(dtype == QSM_F64 || dtype == QSM_F32, "bad dtype");
    QSM_ARG(phas && mask && sz && vsz && uphas && nechoes >= 1, "null pointer or no echo");
    int rc = check_grid(sz, vsz, 1);
    if (rc) return rc;
    const size_t es = dtype_size(dtype), N = sz[0] * sz[1] * sz[2];
    std::vector<char> any[3];
    axis_any(mask, sz, any);
    size_t c0[3], cs[3];
    for (int a = 0; a < 3; ++a) {
        size_t lo = 0, hi = sz[a];
        while (lo < sz[a] && !any[a][lo]) ++lo;
        while (hi > lo && !any[a][hi - 1]) --hi;
        if (lo == hi) {  // empty mask
            std::memset(uphas, 0, N * nechoes * es);
            if (d2phas) std::memset(d2phas, 0, N * nechoes * es);
            return QSM_OK;
        }
        c0[a] = lo > 0 ? lo - 1 : 0;
        cs[a] = std::min(sz[a] - 1, hi) - c0[a] + 1;  // through hi - 1 + 1, clamped
    }
    qsm_mg_opts o;
    qsm_mg_opts_default(&o);
    int L;
    if ((rc = check_mg(dtype, cs, vsz, &o, L))) return rc;
    if ((rc = ensure_device())) return rc;
    const size_t n = cs[0] * cs[1] * cs[2];
    // the crop and the uncrop run on the device: dP and dD hold a whole
    // echo (phase in, then the unwrapped phase; the Laplacian)
    std::vector<int> ix;
    for (int a = 0; a < 3; ++a)
        for (size_t i = 0; i < cs[a]; ++i) ix.push_back(int(c0[a] + i));
    DevBuf dP, dD, dM, dix, du, dm, dout, dd2, dw;
    if ((rc = dP.alloc(N * es)) || (rc = dM.alloc(N)) || (d2phas && (rc = dD.alloc(N * es))) ||
        (rc = dix.alloc(ix.size() * sizeof(int))) || (rc = du.alloc(n * es)) ||
        (rc = dm.alloc(n)) || (rc = dout.alloc(n * es)) || (rc = dd2.alloc(n * es)) ||
        (rc = dw.alloc(qsm_mgpcg_work_bytes(dtype, cs, L))))
        return rc;
    QSM_HIP(hipMemcpy(dM.p, mask, N, hipMemcpyHostToDevice));
    QSM_HIP(hipMemcpy(dix.p, ix.data(), ix.size() * sizeof(int), hipMemcpyHostToDevice));
    const int *dixp = static_cast<const int *>(dix.p);
    const CropMap cm{dixp, dixp + cs[0], dixp + cs[0] + cs[1], int(cs[0]), int(cs[1]),
                     int(cs[2]), sz[0], sz[1], N, n};
    crop_gather_kernel<uint8_t, true><<<crop_blocks(cm, 1), 256>>>(
        static_cast<uint8_t *>(dm.p), static_cast<const uint8_t *>(dM.p), cm, 1);
    QSM_HIP(hipGetLastError());
    // one echo's crop in and out (es bytes per sample)
    auto gather = [&](void *dst, const void *src) {
        if (dtype == QSM_F32)
            crop_gather_kernel<float><<<crop_blocks(cm, 1), 256>>>(
                static_cast<float *>(dst), static_cast<const float *>(src), cm, 1);
        else
            crop_gather_kernel<double><<<crop_blocks(cm, 1), 256>>>(
                static_cast<double *>(dst), static_cast<const double *>(src), cm, 1);
    };
    auto scatter = [&](void *dst, const void *src) {
        if (dtype == QSM_F32)
            crop_scatter_kernel<float><<<crop_blocks(cm, 1), 256>>>(
                static_cast<float *>(dst), static_cast<const float *>(src), cm, 1);
        else
            crop_scatter_kernel<double><<<crop_blocks(cm, 1), 256>>>(
                static_cast<double *>(dst), static_cast<const double *>(src), cm, 1);
    };
    for (size_t e = 0; e < nechoes; ++e) {
        QSM_HIP(hipMemcpy(dP.p, static_cast<const char *>(phas) + e * N * es, N * es,
                          hipMemcpyHostToDevice));
        gather(du.p, dP.p);
        QSM_HIP(hipGetLastError());
        if ((rc = qsm_unwrap_laplacian_dev(dtype, du.p, static_cast<const uint8_t *>(dm.p), cs,
                                           vsz, dout.p, dd2.p, dw.p, nullptr, nullptr)))
            return rc;
        QSM_HIP(hipMemsetAsync(dP.p, 0, N * es, nullptr));
        scatter(dP.p, dout.p);
        if (d2phas) {
            QSM_HIP(hipMemsetAsync(dD.p, 0, N * es, nullptr));
            scatter(dD.p, dd2.p);
        }
        QSM_HIP(hipGetLastError());
        QSM_HIP(hipMemcpy(static_cast<char *>(uphas) + e * N * es, dP.p, N * es,
                          hipMemcpyDeviceToHost));
        if (d2phas)
            QSM_HIP(hipMemcpy(static_cast<char *>(d2phas) + e * N * es, dD.p, N * es,
                              hipMemcpyDeviceToHost));
    }
    return QSM_OK;
}

}  // extern "C"
