// Plasma species on the GPU: initial load, sort by cell, charge deposit,
// psi gather, current/acceleration/momentum-flux deposit and the push.
//
// Particles are a structure of arrays sorted by a tile-major cell key (see
// qp_common.h).  Every particle kernel is cell-centric: one workgroup per
// 16x16-cell tile and one thread per cell.  A thread reads the four corner
// values of the fields its cell needs once, then walks the cell's particles
// (a contiguous run of the sorted arrays), so the per-particle gathers need no
// memory traffic and the per-particle deposits accumulate in registers.  The
// four corner sums of every cell are combined into the tile's 17x17 nodes in
// LDS in a fixed order; nodes inside the tile are written directly and the 64
// border nodes go to a halo buffer that a second kernel sums, again in a fixed
// order, with the one-rank guard fold of PPNACGUARD2L
// (ufield2d_lib.f03:90-97).  No atomics touch the deposits.
#include <hipcub/hipcub.hpp>

#include <cmath>
#include <cstring>
#include <type_traits>

#include "qp_common.h"
#include "qp_border.h"

struct qp_species {
    qp_ctx *ctx;
    qp_species_params p;
    double qbm, dt;
    int64_t np;
    qp::DevBuf a[8], b[8];     // x, y, px, py, pz, p6, p7, q (current, alternate)
    qp::DevBuf key, slot;      // per particle: destination bin and rank (push), key and index (load)
    qp::DevBuf bins;           // per tile: counts, then starts, of the 9 x 256 destination bins
    qp::DevBuf tot;            // particles bound for each tile and group of tiles (push)
    qp::DevBuf count, off;     // per cell (ncells + 1)
    qp::DevBuf off_new;        // the push's new cell offsets, swapped with off
    // every particle has charge q_value (a uniform plasma, or an upload that
    // says so): q is then filled in both buffers and not moved, staged or read
    bool q_uniform;
    double q_value;
    qp::DevBuf scan_tmp, err;
    size_t scan_bytes;
    qp_field2d *q, *qn, *cu, *dcu, *amu;
    // deferred move check of the slice loop: pinned copy of err and its event
    int *h_err;
    hipEvent_t err_ev;
    bool err_pending;
    // piecewise longitudinal density (fdist2d_class.f03:233-251): points
    // s and factors fs; empty for a uniform plasma
    std::vector<double> lp_s, lp_fs;
    double den_factor = 1.0;   // the factor at the last load
    // transverse profile (0 uniform, 10, 11, 12; fdist2d_class.f03:318-950),
    // lengths in grid units
    int profile = 0;
    double pcx = 0, pcy = 0, irx = 0, iry = 0, orx = 0, ory = 0, r0 = 0, sigr = 1;
    std::vector<double> pr, pfr;
    qp::DevBuf radial;         // profile 12: the points pr, then pfr, on the device
};

namespace qp {

template <typename R> struct Soa {
    R *x, *y, *px, *py, *pz, *p6, *p7, *q;
};

template <typename R> static Soa<R> soa(DevBuf *a)
{
    return Soa<R>{a[0].as<R>(), a[1].as<R>(), a[2].as<R>(), a[3].as<R>(),
                  a[4].as<R>(), a[5].as<R>(), a[6].as<R>(), a[7].as<R>()};
}

// Particle positions.  FP64 records hold x and y in grid units, as the
// reference does.  FP32 records hold them relative to the origin of the
// particle's 16 x 16-cell tile (the tile is implied by the sorted order):
// a float near 1000 resolves 6e-5 of a cell, one in [0, 16) 1e-6, and the
// plasma's response ahead of a driver is a displacement of that order per
// slice.  Downloads and uploads convert at the boundary (in FP64), and the
// push re-bases a particle that changes tile.
template <typename R> struct TileRel {
    static constexpr bool on = std::is_same<R, float>::value;
};

// v mod m for -m <= v < 2m (a tile index plus a direction in {-1, 0, 1}):
// the periodic neighbour without an integer division
__device__ __forceinline__ int wrap1(int v, int m) { return v < 0 ? v + m : (v >= m ? v - m : v); }

__host__ __device__ __forceinline__ int cell_key(int cx, int cy, int mx1)
{
    return ((cy >> 4) * mx1 + (cx >> 4)) * TCELLS + ((cy & 15) << 4) + (cx & 15);
}
static inline int host_cell_key(int cx, int cy, int mx1) { return cell_key(cx, cy, mx1); }

// this thread's cell: key = blockIdx.x*256 + threadIdx.x
__device__ __forceinline__ void my_cell(const TileGeom &g, int &cx, int &cy)
{
    int t = blockIdx.x, l = threadIdx.x;
    cx = (t % g.mx1) * TILE + (l & 15);
    cy = (t / g.mx1) * TILE + (l >> 4);
}

template <typename R> struct Corners {
    R f00, f10, f01, f11;
};

template <typename R>
__device__ __forceinline__ Corners<R> load_corners(const R *plane, int ld, int cx, int cy)
{
    const R *r0 = plane + (size_t)cy * ld + cx, *r1 = r0 + ld;
    return Corners<R>{r0[0], r0[1], r1[0], r1[1]};
}

// bilinear gather in the reference's order (e.g. part2d_lib77.f:2265-2268)
template <typename R>
__device__ __forceinline__ R gather(const Corners<R> &f, R amx, R amy, R dxp, R dyp)
{
    R d = amx * f.f00;
    d = amy * (dxp * f.f10 + d);
    R a = amx * f.f01;
    return d + dyp * (dxp * f.f11 + a);
}

template <typename R> static DepOut<R> dep_plain(R *const *planes, int n)
{
    DepOut<R> o{};
    for (int c = 0; c < n; ++c) o.p[c] = planes[c];
    o.scale = o.scale2 = R(1);
    return o;
}

// Sum the tile-border contributions of every border node in a fixed order;
// with fold, row ny is added into row 0 and cleared (PPNACGUARD2L nvp = 1).
// One thread per border node and component (one thread taking every
// component of a node measured 1.5x slower: too few waves per CU).
template <typename R, int RB>
__global__ void k_deposit_border(TileGeom g, const R *__restrict__ halo, size_t halo_cs,
                                 DepOut<R> out, int fold, const int *skip)
{
    if (skip && *skip) return;
    const int comp = blockIdx.y;
    constexpr int B = TILE / RB, SH = RB == 16 ? 4 : RB == 8 ? 3 : 2;
    static_assert(1 << SH == RB, "rows of a block");
    const int myb = g.my1 * B;
    const int rows_n = (myb + 1) * (g.nx + 1);
    const int cols_n = (g.mx1 + 1) * myb * (RB - 1);
    int id = blockIdx.x * blockDim.x + threadIdx.x;
    int X, Y;
    if (id < rows_n) {
        Y = (id / (g.nx + 1)) * RB;
        X = id % (g.nx + 1);
    } else if (id < rows_n + cols_n) {
        int k = id - rows_n;
        int per_col = myb * (RB - 1);
        X = (k / per_col) * TILE;
        int r = k % per_col;
        Y = (r / (RB - 1)) * RB + 1 + r % (RB - 1);
    } else {
        return;
    }
    const R v = border_node<R>(g, halo + comp * halo_cs, SH, fold, X, Y);
    dep_store(out, comp, (size_t)Y * g.ldr + X, v);
}

// LDS slot of staged particle p: one pad word every 32 entries spreads the
// per-cell strided reads over the banks
__device__ __forceinline__ int lpad(int p) { return p + (p >> 5); }

// 1/x: IEEE division in FP64 (the reference's arithmetic); the hardware
// reciprocal (1 ulp) in FP32, whose results are compared with FP64 at 1e-5
__device__ __forceinline__ double recip(double x) { return 1.0 / x; }
__device__ __forceinline__ float recip(float x) { return __builtin_amdgcn_rcpf(x); }
// a / b and sqrt: IEEE in FP64 (the reference's arithmetic); the hardware
// reciprocal and square root (1 ulp) in FP32
__device__ __forceinline__ double divq(double a, double b) { return a / b; }
__device__ __forceinline__ float divq(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
__device__ __forceinline__ double sqrtq(double x) { return sqrt(x); }
__device__ __forceinline__ float sqrtq(float x) { return __builtin_amdgcn_sqrtf(x); }

template <int CH> struct Stage {
    static constexpr int N = CH + CH / 32 + 1;
};

// Stages particles [c0, c0 + n) of NA arrays into LDS (padded index lpad):
// thread tid takes p = tid + k*step, k < K.  Every load of the thread is
// issued before the first LDS store, so the chunk costs one memory latency.
template <typename R, int NA, int K, int M>
__device__ __forceinline__ void stage_in(const R *const (&src)[M], R *const (&dst)[M], int c0,
                                         int n, int tid, int step)
{
    R t[K][NA];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int p = tid + k * step;
        if (p < n) {
#pragma unroll
            for (int a = 0; a < NA; ++a) t[k][a] = src[a][c0 + p];
        }
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int p = tid + k * step;
        if (p < n) {
            const int l = lpad(p);
#pragma unroll
            for (int a = 0; a < NA; ++a) dst[a][l] = t[k][a];
        }
    }
}

// Interior nodes of the tile's 17x17 block to the output plane, border nodes
// to the halo buffer (summed over tiles by k_deposit_border).  With bands, of
// band `band`, RB rows of cells.
template <typename R, int RB = TILE>
__device__ __forceinline__ void emit_nodes(const R *nacc, const DepOut<R> &out, int c, int ldr,
                                           R *halo, int tile, int tx, int ty, int band = 0)
{
    for (int n = threadIdx.x; n < 17 * (RB + 1); n += TCELLS) {
        const int i = n % 17, j = n / 17;
        const R v = nacc[n];
        if (i >= 1 && i < TILE && j >= 1 && j < RB)
            dep_store(out, c, (size_t)(ty * TILE + band * RB + j) * ldr + tx * TILE + i, v);
        else
            halo[(size_t)(tile * (TILE / RB) + band) * band_halo(RB) + halo_index(RB, i, j)] = v;
    }
}

// The same for the eight components of the current deposit, 289 nodes apart in LDS,
// all added to planes (DepOut::inner, no outer).  The planes that are added to are read for all of a node's components before the first
// store: the compiler does not know that the stores leave them alone, and read them
// one after the other.
template <typename R, int RB>
__device__ __forceinline__ void emit_nodes8(const R *nacc, const DepOut<R> &out, int ldr, R *halo,
                                            size_t halo_cs, int tile, int tx, int ty, int band)
{
    for (int n = threadIdx.x; n < 17 * (RB + 1); n += TCELLS) {
        const int i = n % 17, j = n / 17;
        if (i >= 1 && i < TILE && j >= 1 && j < RB) {
            const size_t idx = (size_t)(ty * TILE + band * RB + j) * ldr + tx * TILE + i;
            R in[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) in[c] = out.inner[c][idx];
#pragma unroll
            for (int c = 0; c < 8; ++c) {   // dep_store, with no outer plane
                const R v = nacc[c * 289 + n];
                if (out.p2[c]) out.p2[c][idx] = v * out.scale2;
                out.p[c][idx] = (v + in[c]) * out.scale;
            }
        } else {
            R *h = halo + (size_t)(tile * (TILE / RB) + band) * band_halo(RB) + halo_index(RB, i, j);
#pragma unroll
            for (int c = 0; c < 8; ++c) h[c * halo_cs] = nacc[c * 289 + n];
        }
    }
}

// Deposit skeleton.  The tile's cells are taken RG rows at a time; inside a
// group every cell owns T = 16/RG consecutive lanes (lane cl*T + sub), lane
// sub taking particles sub, sub+T, ... of its cell.  The group's particles
// (a contiguous run of the sorted arrays) are staged through LDS in chunks of
// at most CH with coalesced loads.  Per-lane register sums are reduced over
// the T lanes with xor shuffles and added to the tile's node accumulators in
// four phases (one per cell corner), so every sum has a fixed order and no
// atomic touches the deposit.

// PPGPPOST2L (part2d_lib77.f:194-309): q(n,m) += qm (1-dx)(1-dy) etc.
// UQ: every particle's charge is quni (not staged or read).
// The workgroups past the tiles convert the slice's beam plane (bp), which the
// deposit does not touch: a launch less.
constexpr int BEAM_BLOCKS = 512;
template <typename R, int RG, int CH, int WPE, bool UQ>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE, 8)))
k_deposit_q(TileGeom g, Soa<R> s, const int *__restrict__ off, DepOut<R> out, R *halo, R quni,
            BeamPlane bp)
{
    if ((int)blockIdx.x >= g.mx1 * g.my1) {
        beam_plane_convert<R>(bp, ((size_t)blockIdx.x - g.mx1 * g.my1) * 256 + threadIdx.x,
                              (size_t)BEAM_BLOCKS * 256);
        return;
    }
    constexpr int T = TILE / RG, NP = Stage<CH>::N;
    extern __shared__ unsigned char smem_raw[];
    R *sx = reinterpret_cast<R *>(smem_raw), *sy = sx + NP, *sq = sy + NP, *nacc = UQ ? sq : sq + NP;
    const int tid = threadIdx.x, tile = blockIdx.x;
    const int tx = tile % g.mx1, ty = tile / g.mx1, kb = tile * TCELLS;
    for (int n = tid; n < 289; n += TCELLS) nacc[n] = R(0);
    const int cl = tid / T, sub = tid % T;
    for (int row = 0; row < TILE; row += RG) {
        const int lrow = row + cl / TILE, lcol = cl % TILE;
        const int key = kb + lrow * TILE + lcol;
        const int i0 = off[key], i1 = off[key + 1];
        const int G0 = off[kb + row * TILE], G1 = off[kb + (row + RG) * TILE];
        const R fx = (R)(TileRel<R>::on ? lcol : tx * TILE + lcol);
        const R fy = (R)(TileRel<R>::on ? lrow : ty * TILE + lrow);
        R a00 = 0, a10 = 0, a01 = 0, a11 = 0;
        for (int c0 = G0; c0 < G1; c0 += CH) {
            const int n = min(CH, G1 - c0);
            __syncthreads();
            if (UQ) {
                const R *src[2] = {s.x, s.y};
                R *dst[2] = {sx, sy};
                stage_in<R, 2, CH / TCELLS>(src, dst, c0, n, tid, TCELLS);
            } else {
                const R *src[3] = {s.x, s.y, s.q};
                R *dst[3] = {sx, sy, sq};
                stage_in<R, 3, CH / TCELLS>(src, dst, c0, n, tid, TCELLS);
            }
            __syncthreads();
            int a = i0 + sub;
            if (a < c0) a += ((c0 - a + T - 1) / T) * T;
            const int b = min(i1, c0 + n);
            for (int i = a; i < b; i += T) {
                const int l = lpad(i - c0);
                R qm = UQ ? quni : sq[l];
                R dxp = qm * (sx[l] - fx);
                R dyp = sy[l] - fy;
                R amx = qm - dxp;
                R amy = R(1) - dyp;
                a00 += amx * amy;
                a10 += dxp * amy;
                a01 += amx * dyp;
                a11 += dxp * dyp;
            }
        }
#pragma unroll
        for (int o = T / 2; o > 0; o >>= 1) {
            a00 += __shfl_xor(a00, o);
            a10 += __shfl_xor(a10, o);
            a01 += __shfl_xor(a01, o);
            a11 += __shfl_xor(a11, o);
        }
        const R av[4] = {a00, a10, a01, a11};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            __syncthreads();
            if (sub == 0) nacc[(lrow + (k >> 1)) * 17 + lcol + (k & 1)] += av[k];
        }
    }
    __syncthreads();
    emit_nodes(nacc, out, 0, g.ldr, halo, tile, tx, ty);
}

// Record words 6 and 7 (gamma and gamma - p_z, both 1 for a particle at
// rest).  FP64 stores them as the reference does.  FP32 stores p6 - 1 and
// p7 - 1: a float holding 1 + e keeps e only to 6e-8 absolute, so psi's
// imprint on p7 (e = -qbm psi dex^2) and the p_z formed from p6 and p7 (a
// difference of two numbers near 1/2, part2d_lib77.f:597-598) would carry
// errors of 6e-8/|e| relative, 1e-4 where psi is 1e-3.  The deviations are
// formed without that cancellation and are mathematically the same
// quantities; downloads and uploads convert at the boundary.
template <typename R> struct P67Dev {
    static constexpr bool on = std::is_same<R, float>::value;
};

// WPGPSIPOST2L_QP (part2d_lib77.f:2207-2284): p7 = 1 + dx and
// p6 = dx + (dx2 |v|^2 - dx^2 - 2 dx) / (2 (1 + dx)) + 1 for dx = -qbm psi dex^2;
// in the deviation form p7 - 1 = dx and p6 - 1 = (dx2 |v|^2 + dx^2) / (2 (1 + dx))
template <typename R>
__device__ __forceinline__ void p67_from_psi(R dx, R dx2, R vx, R vy, R &p6, R &p7)
{
    if constexpr (P67Dev<R>::on) {
        p7 = dx;
        p6 = (dx2 * (vx * vx + vy * vy) + dx * dx) / (R(2) * (R(1) + dx));
    } else {
        p7 = R(1) + dx;
        p6 = dx + (dx2 * (vx * vx + vy * vy) - dx * dx - R(2) * dx) / (R(2) * (R(1) + dx)) + R(1);
    }
}

template <typename R>
__global__ void __launch_bounds__(256)
k_extpsi(int64_t np, int nx, int ny, int ldr, Soa<R> s, const R *psi, R qbm, R dex,
         const int *__restrict__ off, int mx1, int ntiles)
{
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= np) return;
    const R x = s.x[i], y = s.y[i];
    int cx, cy;
    R dxp, dyp;
    if constexpr (TileRel<R>::on) {
        // the particle's tile: the last one starting at or before i
        int lo = 0, hi = ntiles - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (off[mid * TCELLS] <= i) lo = mid;
            else hi = mid - 1;
        }
        const int lx = min(max((int)x, 0), TILE - 1), ly = min(max((int)y, 0), TILE - 1);
        cx = (lo % mx1) * TILE + lx;
        cy = (lo / mx1) * TILE + ly;
        dxp = x - (R)lx;
        dyp = y - (R)ly;
    } else {
        cx = min(max((int)x, 0), nx - 1);
        cy = min(max((int)y, 0), ny - 1);
        dxp = x - (R)cx;
        dyp = y - (R)cy;
    }
    const Corners<R> f = load_corners(psi, ldr, cx, cy);
    const R dx2 = dex * dex;
    R amx = R(1) - dxp, amy = R(1) - dyp;
    R vx = s.px[i], vy = s.py[i];
    R dx = gather(f, amx, amy, dxp, dyp);
    dx = -(dx * dx2 * qbm);
    R p6, p7;
    p67_from_psi(dx, dx2, vx, vy, p6, p7);
    s.p7[i] = p7;
    s.p6[i] = p6;
}

// WPGPSIPOST2L_QP for one particle of the cell at (fx, fy): p7 and p6 from
// the psi gather, in k_extpsi's operation order (the first corrector pass
// of a slice applies it just before amjdp_one)
template <typename R>
__device__ __forceinline__ void extpsi_one(const Corners<R> &f, R fx, R fy, R x, R y, R vx, R vy,
                                           R qbm, R dex, R &p6, R &p7)
{
    const R dx2 = dex * dex;
    R dxp = x - fx, dyp = y - fy;
    R amx = R(1) - dxp, amy = R(1) - dyp;
    R dx = gather(f, amx, amy, dxp, dyp);
    dx = -(dx * dx2 * qbm);
    p67_from_psi(dx, dx2, vx, vy, p6, p7);
}

// the six fields amjdp and push gather, at the four corners of one cell
template <typename R> struct Fields6 {
    Corners<R> ex, ey, ez, bx, by, bz;
};

template <typename R>
__device__ __forceinline__ Fields6<R> load_fields6(const R *fxy, const R *bxy, const R *psit,
                                                   size_t cs, int ld, int cx, int cy)
{
    return Fields6<R>{load_corners(fxy, ld, cx, cy),      load_corners(fxy + cs, ld, cx, cy),
                      load_corners(psit, ld, cx, cy),     load_corners(bxy, ld, cx, cy),
                      load_corners(bxy + cs, ld, cx, cy), load_corners(bxy + 2 * cs, ld, cx, cy)};
}

// FP32: a cell's corner values rewritten once as bilinear coefficients,
// f(dxp, dyp) = c0 + dxp c1 + dyp (c2 + dxp c3), so each gather of the cell's
// particles is three FMAs; FP64 keeps the corner values and the reference's
// operation order (gather above)
template <typename R>
__device__ __forceinline__ void prep_fields(Fields6<R> &F)
{
    if constexpr (std::is_same<R, float>::value) {
        Corners<R> *c[6] = {&F.ex, &F.ey, &F.ez, &F.bx, &F.by, &F.bz};
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            const R f00 = c[k]->f00, f10 = c[k]->f10, f01 = c[k]->f01, f11 = c[k]->f11;
            *c[k] = Corners<R>{f00, f10 - f00, f01 - f00, (f11 - f10) - (f01 - f00)};
        }
    }
}

template <typename R>
__device__ __forceinline__ R cell_gather(const Corners<R> &f, R amx, R amy, R dxp, R dyp)
{
    if constexpr (std::is_same<R, float>::value)
        return fmaf(dyp, fmaf(dxp, f.f11, f.f01), fmaf(dxp, f.f10, f.f00));
    else
        return gather(f, amx, amy, dxp, dyp);
}

// One particle of PPGRDCJPPOST2L_QP (part2d_lib77.f:311-768), in the
// reference's operation order: gather, half Boris step with the B_z
// rotation, the 8 deposited quantities times the 4 corner weights added to
// acc; returns the new p6 (part2d_lib77.f:597).
template <typename R>
__device__ __forceinline__ R amjdp_one(const Fields6<R> &F, R fx, R fy, R x, R y, R px, R py,
                                       R p6, R p7, R qm, R qtmh, R qbm, R dti, R dex, R idex,
                                       R (&acc)[8][4])
{
    constexpr bool DEV = P67Dev<R>::on;
    R dxp = x - fx, dyp = y - fy;
    R amx = R(1) - dxp, amy = R(1) - dyp;
    R inv_part_7 = recip(DEV ? R(1) + p7 : p7);
    R qtmh1 = qtmh * inv_part_7;
    R qtmh2 = DEV ? qtmh1 + qtmh1 * p6 : qtmh1 * p6;
    R dx = cell_gather(F.ex, amx, amy, dxp, dyp);
    R dy = cell_gather(F.ey, amx, amy, dxp, dyp);
    R dz = cell_gather(F.ez, amx, amy, dxp, dyp);
    R ox = cell_gather(F.bx, amx, amy, dxp, dyp);
    R oy = cell_gather(F.by, amx, amy, dxp, dyp);
    R oz = cell_gather(F.bz, amx, amy, dxp, dyp);
    R ddx = (R(-1)) * qtmh2 * dx + qtmh * oy;
    R ddy = (R(-1)) * qtmh2 * dy - qtmh * ox;
    R vx = px, vy = py;
    R acx = vx + ddx, acy = vy + ddy;
    R omzt = qtmh1 * oz;
    R omt = omzt * omzt;
    R anorm = R(2) * recip(R(1) + omt);
    R rot1 = R(0.5) * (R(1) - omt);
    R rot2 = omzt;
    R v1 = (rot1 * acx + rot2 * acy) * anorm + ddx;
    R v2 = (rot1 * acy - rot2 * acx) * anorm + ddy;
    R qm1 = qm * inv_part_7;
    amx = qm1 * amx;
    dxp = qm1 * dxp;
    ox = R(0.5) * (v1 + vx);
    oy = R(0.5) * (v2 + vy);
    // p_z = (1 + |p_perp|^2)/(2 p7) - p7/2; with p7 = 1 + e7 it is
    // (|p_perp|^2 - e7 (2 + e7)) / (2 p7), formed without the cancellation
    if constexpr (DEV)
        oz = R(0.5) * (dex * dex * (ox * ox + oy * oy) - p7 * (R(2) + p7)) * inv_part_7;
    else
        oz = R(0.5) * (R(1) + dex * dex * (ox * ox + oy * oy)) * inv_part_7 - R(0.5) * p7;
    const R p6n = p7 + oz;   // gamma = (gamma - p_z) + p_z (both forms)
    oz = oz * idex;
    vx = (v1 - vx) * dti;
    vy = (v2 - vy) * dti;
    dz = qbm * (dz + (dx * ox + dy * oy) * dex * dex * inv_part_7);
    const R w[4] = {amx * amy, dxp * amy, amx * dyp, dxp * dyp};
    v1 = ox * ox * inv_part_7;
    v2 = oy * oy * inv_part_7;
    R v3 = ox * oy * inv_part_7;
    vx = vx + ox * dz * inv_part_7;
    vy = vy + oy * dz * inv_part_7;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        acc[0][k] += ox * w[k];
        acc[1][k] += oy * w[k];
        acc[2][k] += oz * w[k];
        acc[3][k] += vx * w[k];
        acc[4][k] += vy * w[k];
        acc[5][k] += v1 * w[k];
        acc[6][k] += v2 * w[k];
        acc[7][k] += v3 * w[k];
    }
    return p6n;
}

// PPGRDCJPPOST2L_QP (part2d_lib77.f:311-768): half Boris step with the B_z
// rotation, deposit of J (3), dJ/dxi (2) and momentum flux (3); p6 updated.
// PSI = false: a pass without the psi gather (psi is ignored), compiled
// without its corner registers and branches.  (Measured slower: spreading a
// chunk's cells over all four waves at half their lanes, 2 %; each lane
// storing its particles' new p6 itself instead of the copy-back, 1.6 %.)
// UQ: every particle's charge is quni (not staged).
// RG = 0: the rows per group are chosen per tile, as 16 / T for the smallest
// T (lanes per cell: 1, 2, 4, 8 or 16) with which the tile's particles,
// spread evenly over its T groups, stay within THR/4 staging chunks per
// group; a chunk then holds more of its group's cells than with a fixed RG
// in dense tiles (where the lanes of the cells a chunk does not hold wait),
// and a sparse tile takes fewer, larger groups.  (Compiling each T as its
// own path was measured slower: 443-444 against 454.6 slices/s at THR = 4.)
// B: a tile is cut in B bands of rows, one block each (deposit_bands).
// ADD: the sums are added to planes (DepOut::inner), which are read together
// (emit_nodes8).  2048^2, one particle a cell, the deposit and its additions by
// launches of their own, with the stores but a plane at a time, and so: FP32 329,
// 355 and 260 us, FP64 603, 655 and 447.  A kernel of its own: the loads would cost
// the deposits without additions registers (a step at 1024^2 in FP32 4 %).
template <typename R, int RG, int CH, int WPE, bool PSI, bool UQ, int THR = 4, int B = 1,
          bool ADD = false>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE, 8)))
k_amjdp(TileGeom g, Soa<R> s, const int *__restrict__ off, const R *fxy, const R *bxy,
        const R *psit, size_t cs, DepOut<R> out, R *halo, size_t halo_cs, R qbm, R dt, R dex,
        const int *skip, const R *psi_arg, R quni)
{
    const R *psi = PSI ? psi_arg : nullptr;
    if (skip && *skip) return;
    constexpr int NP = Stage<CH>::N;
    extern __shared__ unsigned char smem_raw[];
    R *sx = reinterpret_cast<R *>(smem_raw), *sy = sx + NP, *spx = sy + NP, *spy = spx + NP;
    R *sp6 = spy + NP, *sp7 = sp6 + NP, *sq = sp7 + NP, *nacc = sq + NP;   // nacc: 8 x 289
    constexpr int RB = TILE / B;   // rows of a band
    const int tid = threadIdx.x, tile = (int)blockIdx.x / B, row0 = (int)blockIdx.x % B * RB;
    const int tx = tile % g.mx1, ty = tile / g.mx1, kb = tile * TCELLS;
    for (int n = tid; n < 8 * 289; n += TCELLS) nacc[n] = R(0);
    int T = RG > 0 ? TILE / (RG > 0 ? RG : 1) : B;
    if (RG == 0) {
        const int ntile = off[kb + TCELLS] - off[kb];
        while (T < TILE && 4 * ntile > THR * CH * T) T *= 2;
    }
    const int rg = TILE / T;   // rows per group
    const int cl = tid / T, sub = tid % T;
    const R qtmh = R(0.5) * qbm * dt, dti = R(1) / dt, idex = R(1) / dex;
    for (int row = row0; row < row0 + RB; row += rg) {
        const int lrow = row + cl / TILE, lcol = cl % TILE;
        const int key = kb + lrow * TILE + lcol;
        const int i0 = off[key], i1 = off[key + 1];
        const int G0 = off[kb + row * TILE], G1 = off[kb + (row + rg) * TILE];
        const int cx = tx * TILE + lcol, cy = ty * TILE + lrow;
        Fields6<R> F = load_fields6(fxy, bxy, psit, cs, g.ldr, cx, cy);
        prep_fields(F);
        const Corners<R> FP = psi ? load_corners(psi, g.ldr, cx, cy) : Corners<R>{};
        const R fx = (R)(TileRel<R>::on ? lcol : cx), fy = (R)(TileRel<R>::on ? lrow : cy);
        R acc[8][4];
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[c][k] = R(0);
        for (int c0 = G0; c0 < G1; c0 += CH) {
            const int n = min(CH, G1 - c0);
            __syncthreads();
            // the psi gather makes p6 and p7 anew: they are not read (1024^2, 16 a
            // cell: FP32 178 -> 163 us, FP64 372 -> 350)
            constexpr int NS = PSI ? 4 : 6;
            if (UQ) {
                const R *src[6] = {s.x, s.y, s.px, s.py, s.p6, s.p7};
                R *dst[6] = {sx, sy, spx, spy, sp6, sp7};
                stage_in<R, NS, CH / TCELLS>(src, dst, c0, n, tid, TCELLS);
            } else {
                const R *src[7] = {s.x, s.y, s.px, s.py, PSI ? s.q : s.p6, s.p7, s.q};
                R *dst[7] = {sx, sy, spx, spy, PSI ? sq : sp6, sp7, sq};
                stage_in<R, NS + 1, CH / TCELLS>(src, dst, c0, n, tid, TCELLS);
            }
            __syncthreads();
            int a = i0 + sub;
            if (a < c0) a += ((c0 - a + T - 1) / T) * T;
            const int b = min(i1, c0 + n);
            for (int i = a; i < b; i += T) {
                const int l = lpad(i - c0);
                R p6 = PSI ? R(0) : sp6[l], p7 = PSI ? R(0) : sp7[l];
                if (psi) {
                    extpsi_one(FP, fx, fy, sx[l], sy[l], spx[l], spy[l], qbm, dex, p6, p7);
                    sp7[l] = p7;
                }
                sp6[l] = amjdp_one(F, fx, fy, sx[l], sy[l], spx[l], spy[l], p6, p7,
                                   UQ ? quni : sq[l], qtmh, qbm, dti, dex, idex, acc);
            }
            __syncthreads();
            for (int p = tid; p < n; p += TCELLS) s.p6[c0 + p] = sp6[lpad(p)];
            if (psi)
                for (int p = tid; p < n; p += TCELLS) s.p7[c0 + p] = sp7[lpad(p)];
        }
        for (int o = T / 2; o > 0; o >>= 1)
#pragma unroll
            for (int c = 0; c < 8; ++c)
#pragma unroll
                for (int k = 0; k < 4; ++k) acc[c][k] += __shfl_xor(acc[c][k], o);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            __syncthreads();
            if (sub == 0) {
                const int node = (lrow - row0 + (k >> 1)) * 17 + lcol + (k & 1);
#pragma unroll
                for (int c = 0; c < 8; ++c) nacc[c * 289 + node] += acc[c][k];
            }
        }
    }
    __syncthreads();
    if (ADD) {
        emit_nodes8<R, RB>(nacc, out, g.ldr, halo, halo_cs, tile, tx, ty, row0 / RB);
        return;
    }
#pragma unroll
    for (int c = 0; c < 8; ++c)
        emit_nodes<R, RB>(nacc + c * 289, out, c, g.ldr, halo + c * halo_cs, tile, tx, ty,
                          row0 / RB);
}

// The same deposit with the next chunk's particles loaded into registers
// while the current chunk is computed, so a workgroup's global loads overlap
// its own arithmetic (the staging chunk of k_amjdp waits for its loads).
// The tile's particles are one contiguous run, row group after row group, so
// the chunk after the last of a group is the first of the next; a chunk that
// was not prefetched (after an empty group) is loaded when it is reached.
// Cells, lanes, sums and their order are those of k_amjdp with the same RG.
template <typename R, int RG, int CH>
__global__ void __launch_bounds__(256)
k_amjdp_pf(TileGeom g, Soa<R> s, const int *__restrict__ off, const R *fxy, const R *bxy,
           const R *psit, size_t cs, DepOut<R> out, R *halo, size_t halo_cs, R qbm, R dt, R dex,
           const int *skip, const R *psi, R)
{
    if (skip && *skip) return;
    constexpr int T = TILE / RG, NP = Stage<CH>::N, PF = CH / TCELLS;
    extern __shared__ unsigned char smem_raw[];
    R *sx = reinterpret_cast<R *>(smem_raw), *sy = sx + NP, *spx = sy + NP, *spy = spx + NP;
    R *sp6 = spy + NP, *sp7 = sp6 + NP, *sq = sp7 + NP, *nacc = sq + NP;   // nacc: 8 x 289
    const int tid = threadIdx.x, tile = blockIdx.x;
    const int tx = tile % g.mx1, ty = tile / g.mx1, kb = tile * TCELLS;
    for (int n = tid; n < 8 * 289; n += TCELLS) nacc[n] = R(0);
    const int cl = tid / T, sub = tid % T;
    const R qtmh = R(0.5) * qbm * dt, dti = R(1) / dt, idex = R(1) / dex;
    R rx[PF], ry[PF], rpx[PF], rpy[PF], rp6[PF], rp7[PF], rq[PF];
    int pc0 = -1, pn = 0;   // the chunk held in the registers
    auto fetch = [&](int b0, int nn) {
#pragma unroll
        for (int k = 0; k < PF; ++k) {
            const int p = tid + k * TCELLS;
            if (p < nn) {
                const int q = b0 + p;
                rx[k] = s.x[q];
                ry[k] = s.y[q];
                rpx[k] = s.px[q];
                rpy[k] = s.py[q];
                rp6[k] = s.p6[q];
                rp7[k] = s.p7[q];
                rq[k] = s.q[q];
            }
        }
        pc0 = b0;
        pn = nn;
    };
    for (int row = 0; row < TILE; row += RG) {
        const int lrow = row + cl / TILE, lcol = cl % TILE;
        const int key = kb + lrow * TILE + lcol;
        const int i0 = off[key], i1 = off[key + 1];
        const int G0 = off[kb + row * TILE], G1 = off[kb + (row + RG) * TILE];
        const int G2 = row + RG < TILE ? off[kb + (row + 2 * RG) * TILE] : G1;
        const int cx = tx * TILE + lcol, cy = ty * TILE + lrow;
        Fields6<R> F = load_fields6(fxy, bxy, psit, cs, g.ldr, cx, cy);
        prep_fields(F);
        const Corners<R> FP = psi ? load_corners(psi, g.ldr, cx, cy) : Corners<R>{};
        const R fx = (R)(TileRel<R>::on ? lcol : cx), fy = (R)(TileRel<R>::on ? lrow : cy);
        R acc[8][4];
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[c][k] = R(0);
        for (int c0 = G0; c0 < G1; c0 += CH) {
            const int n = min(CH, G1 - c0);
            if (pc0 != c0 || pn != n) fetch(c0, n);
            __syncthreads();
#pragma unroll
            for (int k = 0; k < PF; ++k) {
                const int p = tid + k * TCELLS;
                if (p < n) {
                    const int l = lpad(p);
                    sx[l] = rx[k];
                    sy[l] = ry[k];
                    spx[l] = rpx[k];
                    spy[l] = rpy[k];
                    sp6[l] = rp6[k];
                    sp7[l] = rp7[k];
                    sq[l] = rq[k];
                }
            }
            __syncthreads();
            // the next chunk: the rest of this group, or the start of the next
            const int nc0 = c0 + n;
            const int nn = nc0 < G1 ? min(CH, G1 - nc0) : min(CH, G2 - nc0);
            if (nn > 0) fetch(nc0, nn);
            else pc0 = -1;
            int a = i0 + sub;
            if (a < c0) a += ((c0 - a + T - 1) / T) * T;
            const int b = min(i1, c0 + n);
            for (int i = a; i < b; i += T) {
                const int l = lpad(i - c0);
                R p6 = sp6[l], p7 = sp7[l];
                if (psi) {
                    extpsi_one(FP, fx, fy, sx[l], sy[l], spx[l], spy[l], qbm, dex, p6, p7);
                    sp7[l] = p7;
                }
                sp6[l] = amjdp_one(F, fx, fy, sx[l], sy[l], spx[l], spy[l], p6, p7, sq[l], qtmh,
                                   qbm, dti, dex, idex, acc);
            }
            __syncthreads();
            for (int p = tid; p < n; p += TCELLS) s.p6[c0 + p] = sp6[lpad(p)];
            if (psi)
                for (int p = tid; p < n; p += TCELLS) s.p7[c0 + p] = sp7[lpad(p)];
        }
#pragma unroll
        for (int o = T / 2; o > 0; o >>= 1)
#pragma unroll
            for (int c = 0; c < 8; ++c)
#pragma unroll
                for (int k = 0; k < 4; ++k) acc[c][k] += __shfl_xor(acc[c][k], o);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            __syncthreads();
            if (sub == 0) {
                const int node = (lrow + (k >> 1)) * 17 + lcol + (k & 1);
#pragma unroll
                for (int c = 0; c < 8; ++c) nacc[c * 289 + node] += acc[c][k];
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 8; ++c)
        emit_nodes(nacc + c * 289, out, c, g.ldr, halo + c * halo_cs, tile, tx, ty);
}

// FP32 deposit with the particle chunks copied from memory into LDS by the
// LDS-DMA loads (global_load_lds_dword: each lane's dword lands at the wave's
// LDS base + 4 lane) into two buffers: the next chunk is in flight while the
// current one is computed, and the copy uses no registers.  Chunks hold CH
// particles; LDS index of particle p of a chunk: p + p/64 (one pad per
// wave block).  Cells, lanes, sums and their order are those of k_amjdp.
__device__ __forceinline__ int lpad64(int p) { return p + (p >> 6); }

template <int RG, int CH>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 8)))
k_amjdp_dma(TileGeom g, Soa<float> s, const int *__restrict__ off, const float *fxy,
            const float *bxy, const float *psit, size_t cs, DepOut<float> out, float *halo,
            size_t halo_cs, float qbm, float dt, float dex, const int *skip, const float *psi,
            float)
{
    using R = float;
    if (skip && *skip) return;
    constexpr int T = TILE / RG, NB = CH + CH / 64, K = CH / TCELLS;
    extern __shared__ unsigned char smem_raw[];
    R *base = reinterpret_cast<R *>(smem_raw);          // [2 buffers][7 arrays][NB]
    R *nacc = base + 2 * 7 * NB;                         // 8 x 289
    const int tid = threadIdx.x, tile = blockIdx.x, lane = tid & 63, wave = tid >> 6;
    const int tx = tile % g.mx1, ty = tile / g.mx1, kb = tile * TCELLS;
    for (int n = tid; n < 8 * 289; n += TCELLS) nacc[n] = R(0);
    const int cl = tid / T, sub = tid % T;
    const R qtmh = R(0.5) * qbm * dt, dti = R(1) / dt, idex = R(1) / dex;
    const R *src[7] = {s.x, s.y, s.px, s.py, s.p6, s.p7, s.q};
    // copy chunk [b0, b0 + nn) into buffer bf: wave w takes blocks k*256 + 64 w
    auto issue = [&](int b0, int nn, int bf) {
#pragma unroll
        for (int a = 0; a < 7; ++a) {
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const int blk = k * TCELLS + wave * 64;
                if (blk + lane < nn)
                    __builtin_amdgcn_global_load_lds(
                        src[a] + b0 + blk + lane,
                        (__attribute__((address_space(3))) void *)(base + (bf * 7 + a) * NB +
                                                                   lpad64(blk)),
                        4, 0, 0);
            }
        }
    };
    int pc0 = -1, pn = 0, cur = 0;
    for (int row = 0; row < TILE; row += RG) {
        const int lrow = row + cl / TILE, lcol = cl % TILE;
        const int key = kb + lrow * TILE + lcol;
        const int i0 = off[key], i1 = off[key + 1];
        const int G0 = off[kb + row * TILE], G1 = off[kb + (row + RG) * TILE];
        const int G2 = row + RG < TILE ? off[kb + (row + 2 * RG) * TILE] : G1;
        const int cx = tx * TILE + lcol, cy = ty * TILE + lrow;
        Fields6<R> F = load_fields6(fxy, bxy, psit, cs, g.ldr, cx, cy);
        prep_fields(F);
        const Corners<R> FP = psi ? load_corners(psi, g.ldr, cx, cy) : Corners<R>{};
        const R fx = (R)(TileRel<R>::on ? lcol : cx), fy = (R)(TileRel<R>::on ? lrow : cy);
        R acc[8][4];
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[c][k] = R(0);
        for (int c0 = G0; c0 < G1; c0 += CH) {
            const int n = min(CH, G1 - c0);
            if (pc0 != c0 || pn != n) issue(c0, n, cur);
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            // the next chunk: the rest of this group, or the start of the next
            const int nc0 = c0 + n;
            const int nn = nc0 < G1 ? min(CH, G1 - nc0) : min(CH, G2 - nc0);
            if (nn > 0) {
                issue(nc0, nn, cur ^ 1);
                pc0 = nc0;
                pn = nn;
            } else {
                pc0 = -1;
            }
            R *sx = base + (cur * 7 + 0) * NB, *sy = sx + NB, *spx = sy + NB, *spy = spx + NB;
            R *sp6 = spy + NB, *sp7 = sp6 + NB, *sq = sp7 + NB;
            int a = i0 + sub;
            if (a < c0) a += ((c0 - a + T - 1) / T) * T;
            const int b = min(i1, c0 + n);
            for (int i = a; i < b; i += T) {
                const int l = lpad64(i - c0);
                R p6 = sp6[l], p7 = sp7[l];
                if (psi) {
                    extpsi_one(FP, fx, fy, sx[l], sy[l], spx[l], spy[l], qbm, dex, p6, p7);
                    sp7[l] = p7;
                }
                sp6[l] = amjdp_one(F, fx, fy, sx[l], sy[l], spx[l], spy[l], p6, p7, sq[l], qtmh,
                                   qbm, dti, dex, idex, acc);
            }
            __syncthreads();
            for (int p = tid; p < n; p += TCELLS) s.p6[c0 + p] = sp6[lpad64(p)];
            if (psi)
                for (int p = tid; p < n; p += TCELLS) s.p7[c0 + p] = sp7[lpad64(p)];
            cur ^= 1;
        }
#pragma unroll
        for (int o = T / 2; o > 0; o >>= 1)
#pragma unroll
            for (int c = 0; c < 8; ++c)
#pragma unroll
                for (int k = 0; k < 4; ++k) acc[c][k] += __shfl_xor(acc[c][k], o);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            __syncthreads();
            if (sub == 0) {
                const int node = (lrow + (k >> 1)) * 17 + lcol + (k & 1);
#pragma unroll
                for (int c = 0; c < 8; ++c) nacc[c * 289 + node] += acc[c][k];
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 8; ++c)
        emit_nodes(nacc + c * 289, out, c, g.ldr, halo + c * halo_cs, tile, tx, ty);
}

// Orders LDS accesses among the lanes of one wave (no workgroup barrier).
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The same deposit with the waves of a tile working independently: wave w
// takes the tile's row pairs w and w+4 (32 cells, two lanes per cell),
// stages that pair's particles through its own LDS area in chunks of CHW,
// and adds its cell sums into its own 3 x 17 node rows in four corner phases
// (wave-level ordering only).  One workgroup barrier at the end, then each
// tile node is the sum, in row-pair order, of the (one or two) row-pair node
// rows that hold it.  A heavy row pair delays only its own wave.
template <typename R, int CHW>
__global__ void __launch_bounds__(256)
k_amjdp_w(TileGeom g, Soa<R> s, const int *__restrict__ off, const R *fxy, const R *bxy,
          const R *psit, size_t cs, DepOut<R> out, R *halo, size_t halo_cs, R qbm, R dt, R dex,
          const int *skip, const R *psi, R)
{
    if (skip && *skip) return;
    constexpr int NP = Stage<CHW>::N, NR = 3 * 17;   // node rows of a row pair
    extern __shared__ unsigned char smem_raw[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    R *base = reinterpret_cast<R *>(smem_raw);
    R *sx = base + wave * 7 * NP, *sy = sx + NP, *spx = sy + NP, *spy = spx + NP;
    R *sp6 = spy + NP, *sp7 = sp6 + NP, *sq = sp7 + NP;
    R *rnode = base + 4 * 7 * NP;                     // [row pair 8][comp 8][3][17]
    const int tile = blockIdx.x, tx = tile % g.mx1, ty = tile / g.mx1, kb = tile * TCELLS;
    for (int n = tid; n < 8 * 8 * NR; n += TCELLS) rnode[n] = R(0);
    __syncthreads();
    const int cl = lane >> 1, sub = lane & 1;
    const R qtmh = R(0.5) * qbm * dt, dti = R(1) / dt, idex = R(1) / dex;
    for (int it = 0; it < 2; ++it) {
        const int rp = wave + 4 * it;
        const int lrow = 2 * rp + (cl >> 4), lcol = cl & 15;
        const int key = kb + lrow * TILE + lcol;
        const int i0 = off[key], i1 = off[key + 1];
        const int G0 = off[kb + 2 * rp * TILE], G1 = off[kb + (2 * rp + 2) * TILE];
        const int cx = tx * TILE + lcol, cy = ty * TILE + lrow;
        Fields6<R> F = load_fields6(fxy, bxy, psit, cs, g.ldr, cx, cy);
        prep_fields(F);
        const Corners<R> FP = psi ? load_corners(psi, g.ldr, cx, cy) : Corners<R>{};
        const R fx = (R)(TileRel<R>::on ? lcol : cx), fy = (R)(TileRel<R>::on ? lrow : cy);
        R acc[8][4];
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[c][k] = R(0);
        for (int c0 = G0; c0 < G1; c0 += CHW) {
            const int n = min(CHW, G1 - c0);
            wave_sync();
            {
                const R *src[7] = {s.x, s.y, s.px, s.py, s.p6, s.p7, s.q};
                R *dst[7] = {sx, sy, spx, spy, sp6, sp7, sq};
                stage_in<R, 7, CHW / 64>(src, dst, c0, n, lane, 64);
            }
            wave_sync();
            int a = i0 + sub;
            if (a < c0) a += ((c0 - a + 1) / 2) * 2;
            const int b = min(i1, c0 + n);
            for (int i = a; i < b; i += 2) {
                const int l = lpad(i - c0);
                R p6 = sp6[l], p7 = sp7[l];
                if (psi) {
                    extpsi_one(FP, fx, fy, sx[l], sy[l], spx[l], spy[l], qbm, dex, p6, p7);
                    sp7[l] = p7;
                }
                sp6[l] = amjdp_one(F, fx, fy, sx[l], sy[l], spx[l], spy[l], p6, p7, sq[l], qtmh,
                                   qbm, dti, dex, idex, acc);
            }
            wave_sync();
            for (int p = lane; p < n; p += 64) s.p6[c0 + p] = sp6[lpad(p)];
            if (psi)
                for (int p = lane; p < n; p += 64) s.p7[c0 + p] = sp7[lpad(p)];
        }
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[c][k] += __shfl_xor(acc[c][k], 1);
        R *rn = rnode + rp * 8 * NR;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            wave_sync();
            if (sub == 0) {
                const int node = ((cl >> 4) + (k >> 1)) * 17 + lcol + (k & 1);
#pragma unroll
                for (int c = 0; c < 8; ++c) rn[c * NR + node] += acc[c][k];
            }
        }
    }
    __syncthreads();
    for (int n = tid; n < 17 * 17; n += TCELLS) {
        const int i = n % 17, j = n / 17;
        const int rp = j >> 1;                 // row pair whose node row j%2 is node row j
        const bool top = (j & 1) == 0 && j > 0;   // also row 2 of row pair rp-1
        for (int c = 0; c < 8; ++c) {
            R v;
            if (j == 16) v = rnode[(7 * 8 + c) * NR + 2 * 17 + i];
            else {
                v = rnode[(rp * 8 + c) * NR + (j & 1) * 17 + i];
                if (top) v = rnode[((rp - 1) * 8 + c) * NR + 2 * 17 + i] + v;
            }
            if (i >= 1 && i < TILE && j >= 1 && j < TILE)
                dep_store(out, c, (size_t)(ty * TILE + j) * g.ldr + tx * TILE + i, v);
            else
                halo[c * halo_cs + (size_t)tile * HALO + halo_index(TILE, i, j)] = v;
        }
    }
}

// PPGRBPPUSHF23L_QP (part2d_lib77.f:1066-1408): 3-D Boris push in xi, then the
// periodic wrap of the reorder (PPPORDER2LB :1936-1977).  One workgroup per
// source tile walks the tile's particles (a contiguous run of the sorted
// arrays) NT at a time, one thread per particle.  A particle leaves for the
// neighbour tile in its direction of motion (dir in {-1,0,1}^2, bin
// nb = 3 (diry+1) + dirx + 1) and lands in cell cl of it; its rank among the
// tile's particles bound for the same (nb, cl) follows their order in the
// tile: lanes of a wave rank by lane order, and a wave counts the earlier waves'
// particles of its bins in the chunk (a byte each) and the earlier chunks' (the
// tile's LDS histogram).  So the new order is a function of the old one: the
// sort, and with it every later sum, is the same run to run.  (A wave finding
// its equal bins one bin after the other, and the waves updating the histogram
// in turn, took 26.9 us against 19.3 us at 512^2, 212 against 204 at 1024^2, where
// it moves its bytes at 4.6 TB/s.)  The histogram goes to cnt[tile][nb][cl].  A particle whose new
// tile is not its old tile plus its direction (the condition PPPCHECK2L
// reports) sets *err and is kept in its own tile.
//
// MODE 0 stores the pushed particle in place with its bin and rank (k_scatter
// then moves it).  MODE 1 stores nothing per particle: only the histogram,
// counted with LDS integer atomics (the same counts in any order; no ranks).
// MODE 2 runs after MODE 1 and k_bin_offsets, which turns cnt into each bin's
// start within its cell and fills off_new: it repeats the push on the unchanged
// input, so bins and ranks are those of MODE 1, and stores each particle at
// off_new[cell] + start + rank of the alternate arrays o.  raw: fxy holds
// grad(psi) still, and the gathered E_perp is formed from it and B_perp
// (efield_x, efield_y).  tot (MODE 1): the particles bound for every tile, summed
// for k_bin_offsets (one atomic per neighbour that gets any: one per wave and
// group of tiles took 80 us more at 1024^2); MODE 2 clears them for the next push.
// The two passes read the particle record twice and write it once, where push and
// scatter read it twice and write it twice.
constexpr int NBINS = 9 * TCELLS;
constexpr int PUSH_WIDE = 1024;   // threads of a block where tiles are few (push_t)
constexpr int BIN_BITS = 12;
static_assert(NBINS <= 1 << BIN_BITS && TCELLS / 64 == 4, "push: bins and waves");
constexpr int GROUP = 256;  // tiles per group of the offsets' two-level sum

template <typename R, int MODE, int NT = 256>
__global__ void __launch_bounds__(NT)
k_push(TileGeom g, Soa<R> s, Soa<R> o, const int *__restrict__ off,
       const int *__restrict__ off_new, const R *fxy, const R *bxy, const R *psit, size_t cs,
       R qbm, R dt, R dex, int *bin, int *rank, int *cnt, int *err, int64_t np, int uq, int raw,
       int *tot)
{
    __shared__ int hist[NBINS];
    // byte w of a bin: wave w's particles in this chunk
    constexpr int NW = NT / 64;
    __shared__ __attribute__((aligned(16))) unsigned whist[MODE == 1 ? 1 : NBINS * NW / 4];
    __shared__ R fnode[6][289];   // the six fields at the tile's 17 x 17 nodes
    const int S = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int k = tid; k < NBINS; k += NT) hist[k] = 0;
    if (MODE != 1)
        for (int k = tid; k < NBINS * NW / 4; k += NT) whist[k] = 0;
    const int tx0 = S % g.mx1, ty0 = S / g.mx1;
    const int p0 = off[S * TCELLS], p1 = off[(S + 1) * TCELLS];
    // the particle record of chunk c0 is loaded while chunk c0 - NT is ranked
    R nx_ = R(0), ny_ = R(0), npx = R(0), npy = R(0), npz = R(0), np6 = R(1), np7 = R(1);
    R nq = R(0);
    auto fetch = [&](int c) {
        const int i = c + tid;
        if (i < p1) {
            nx_ = s.x[i];
            ny_ = s.y[i];
            npx = s.px[i];
            npy = s.py[i];
            npz = s.pz[i];
            np6 = s.p6[i];
            np7 = s.p7[i];
            if (MODE == 2 && !uq) nq = s.q[i];
        }
    };
    fetch(p0);
    // every particle of the tile lies in one of its cells (the sort put it
    // there), so the corners it gathers are tile nodes: read them once
    {
        constexpr int NF = (6 * 289 + NT - 1) / NT;
        R tv[NF];
#pragma unroll
        for (int k = 0; k < NF; ++k) {
            const int n = tid + k * NT;
            if (n < 6 * 289) {
                const int f = n / 289, m = n % 289;
                const R *pl = f == 0 ? fxy : f == 1 ? fxy + cs : f == 2 ? psit
                            : f == 3 ? bxy : f == 4 ? bxy + cs : bxy + 2 * cs;
                const size_t o = (size_t)(ty0 * TILE + m / 17) * g.ldr + tx0 * TILE + m % 17;
                tv[k] = pl[o];
                if (raw && f < 2)
                    tv[k] = f == 0 ? efield_x(tv[k], bxy[cs + o]) : efield_y(tv[k], bxy[o]);
            }
        }
#pragma unroll
        for (int k = 0; k < NF; ++k) {
            const int n = tid + k * NT;
            if (n < 6 * 289) fnode[n / 289][n % 289] = tv[k];
        }
    }
    __syncthreads();
    const R idex = R(1) / dex, qtmh = R(0.5) * qbm * dt;
    const R anx = (R)g.nx, any = (R)g.ny;
    const R edgelx = (R)(tx0 * TILE), edgely = (R)(ty0 * TILE);
    const R edgerx = edgelx + (R)min(TILE, g.nx - tx0 * TILE);
    const R edgery = edgely + (R)min(TILE, g.ny - ty0 * TILE);
    for (int c0 = p0; c0 < p1; c0 += NT) {
        const int i = c0 + tid;
        const bool valid = i < p1;
        const R x = nx_, y = ny_, ppx = npx, ppy = npy, ppz = npz, p6 = np6, p7 = np7, q = nq;
        if (c0 + NT < p1) fetch(c0 + NT);
        int b = 0, dcell = 0;
        R ox_ = R(0), oy_ = R(0), opx = R(0), opy = R(0), opz = R(0);
        if (valid) {
            // absolute cell (FP64) or cell within the tile (FP32 tile-relative)
            const int cx = TileRel<R>::on ? min(max((int)x, 0), TILE - 1)
                                          : min(max((int)x, 0), g.nx - 1);
            const int cy = TileRel<R>::on ? min(max((int)y, 0), TILE - 1)
                                          : min(max((int)y, 0), g.ny - 1);
            // local node of the cell, clamped into the tile (a particle flagged
            // by the move check may sit outside it; its result is reported)
            const int li = TileRel<R>::on ? cx : min(max(cx - tx0 * TILE, 0), TILE - 1);
            const int lj = TileRel<R>::on ? cy : min(max(cy - ty0 * TILE, 0), TILE - 1);
            const int m = lj * 17 + li;
            auto lc = [&](int f) {
                return Corners<R>{fnode[f][m], fnode[f][m + 1], fnode[f][m + 17], fnode[f][m + 18]};
            };
            const Corners<R> ex = lc(0), ey = lc(1), ez = lc(2), bx = lc(3), by = lc(4), bz = lc(5);
            R qtmh1 = divq(qtmh, P67Dev<R>::on ? R(1) + p7 : p7);
            R qtmh2 = P67Dev<R>::on ? qtmh1 + qtmh1 * p6 : qtmh1 * p6;
            R dxp = x - (R)cx, dyp = y - (R)cy;
            R amx = R(1) - dxp, amy = R(1) - dyp;
            R dx = gather(ex, amx, amy, dxp, dyp);
            R dy = gather(ey, amx, amy, dxp, dyp);
            R dz = gather(ez, amx, amy, dxp, dyp);
            dz = dz * idex;
            R ox = gather(bx, amx, amy, dxp, dyp);
            R oy = gather(by, amx, amy, dxp, dyp);
            R oz = gather(bz, amx, amy, dxp, dyp);
            ox = ox * dex;
            oy = oy * dex;
            dx = qtmh2 * dx;
            dy = qtmh2 * dy;
            dz = qtmh2 * dz;
            R acx = ppx + dx, acy = ppy + dy, acz = ppz + dz;
            R omxt = qtmh1 * ox, omyt = qtmh1 * oy, omzt = qtmh1 * oz;
            R omt = omxt * omxt + omyt * omyt + omzt * omzt;
            R anorm = divq(R(2), R(1) + omt);
            omt = R(0.5) * (R(1) - omt);
            R rot4 = omxt * omyt, rot7 = omxt * omzt, rot8 = omyt * omzt;
            R rot1 = omt + omxt * omxt;
            R rot5 = omt + omyt * omyt;
            R rot9 = omt + omzt * omzt;
            R rot2 = omzt + rot4;
            rot4 = -omzt + rot4;
            R rot3 = -omyt + rot7;
            rot7 = omyt + rot7;
            R rot6 = omxt + rot8;
            rot8 = -omxt + rot8;
            dx = (rot1 * acx + rot2 * acy + rot3 * acz) * anorm + dx;
            dy = (rot4 * acx + rot5 * acy + rot6 * acz) * anorm + dy;
            dz = (rot7 * acx + rot8 * acy + rot9 * acz) * anorm + dz;
            if (MODE == 0) {
                s.px[i] = dx;
                s.py[i] = dy;
                s.pz[i] = dz;
            }
            opx = dx;
            opy = dy;
            opz = dz;
            R dtc1 = divq(dt, sqrtq(R(1) + (dx * dx + dy * dy + dz * dz) * dex * dex) - dz * dex);
            dx = x + dx * dtc1;
            dy = y + dy * dtc1;
            int dirx = 0, diry = 0, ncx, ncy;
            bool far = false;   // beyond the neighbouring tiles (PPPCHECK2L)
            if constexpr (TileRel<R>::on) {
                // A position that leaves [0, 16) moves to the neighbouring
                // tile and is re-based by 16 (exact for -16 <= x < 32).  One
                // just below 0 whose re-based value rounds to 16 stays at 0,
                // as the absolute form keeps a particle whose wrap rounds to
                // the box edge.  Tile indices wrap periodically below.
                const R T = (R)TILE;
                if (dx >= T) { dirx = 1; dx = dx - T; }
                else if (dx < R(0)) {
                    if (dx + T >= T) dx = R(0);
                    else { dirx = -1; dx = dx + T; }
                }
                if (dy >= T) { diry = 1; dy = dy - T; }
                else if (dy < R(0)) {
                    if (dy + T >= T) dy = R(0);
                    else { diry = -1; dy = dy + T; }
                }
                far = !(dx >= R(0) && dx < T && dy >= R(0) && dy < T);
                if (far && !(isfinite(dx) && isfinite(dy)) && MODE != 2) atomicMax(err, 1 << 30);
                ncx = far ? min(max((int)dx, 0), TILE - 1) : (int)dx;
                ncy = far ? min(max((int)dy, 0), TILE - 1) : (int)dy;
            } else {
                if (dx >= edgerx) dirx = 1;
                else if (dx < edgelx) {
                    dirx = -1;
                    if (dx < R(0) && dx + anx >= anx) { dx = R(0); dirx = 0; }
                }
                if (dy >= edgery) diry = 1;
                else if (dy < edgely) {
                    diry = -1;
                    if (dy < R(0) && dy + any >= any) { dy = R(0); diry = 0; }
                }
                if (dx < R(0)) dx = dx + anx;
                if (dx >= anx) dx = dx - anx;
                if (dy < R(0)) dy = dy + any;
                if (dy >= any) dy = dy - any;
                ncx = (int)dx;
                ncy = (int)dy;
                // a non-finite or out-of-range position must not become an index
                if (!(ncx >= 0 && ncx < g.nx && ncy >= 0 && ncy < g.ny)) {
                    if (MODE != 2) atomicMax(err, 1 << 30);
                    ncx = min(max(ncx, 0), g.nx - 1);
                    ncy = min(max(ncy, 0), g.ny - 1);
                }
            }
            if (MODE == 0) {
                s.x[i] = dx;
                s.y[i] = dy;
            }
            ox_ = dx;
            oy_ = dy;
            const int txd = wrap1(tx0 + dirx, g.mx1), tyd = wrap1(ty0 + diry, g.my1);
            // destination tile: the neighbour in the direction of motion, or,
            // for a particle the move check flags, its own tile
            int dt = tyd * g.mx1 + txd;
            if (!TileRel<R>::on) far = (ncx >> 4) != txd || (ncy >> 4) != tyd;
            if (far) {
                if (MODE != 2) atomicMax(err, 1 + txd + g.mx1 * tyd);
                dirx = diry = 0;
                dt = S;
            }
            b = (3 * (diry + 1) + dirx + 1) * TCELLS + ((ncy & 15) << 4) + (ncx & 15);
            dcell = dt * TCELLS + (b & 255);
        }
        if (MODE == 1) {
            // counting only (integer adds give the same counts in any order):
            // one LDS atomic per run of equal bins along the lanes, of the
            // run's length (valid lanes are a prefix of the wave)
            const int bprev = __shfl_up(b, 1);
            const bool head = valid && (lane == 0 || bprev != b);
            const unsigned long long heads = __ballot(head);
            const int nvalid = __popcll(__ballot(valid));
            const unsigned long long above = heads & ~((2ull << lane) - 1ull);
            const int end = above ? __ffsll((long long)above) - 1 : nvalid;
            if (head) atomicAdd(&hist[b], end - lane);
            continue;
        }
        // rank among the wave's earlier particles of the same bin: the lanes whose
        // bin agrees in every bit
        unsigned long long m = __ballot(valid);
#pragma unroll
        for (int k = 0; k < BIN_BITS; ++k) {
            const bool bit = (b >> k) & 1;
            const unsigned long long set = __ballot(bit);
            m &= bit ? set : ~set;
        }
        int rk = __popcll(m & ((1ull << lane) - 1ull));
        const bool lead = valid && rk == 0;
        const int nlead = __popcll(m);   // at most 64
        if (lead) reinterpret_cast<unsigned char *>(whist)[NW * b + wave] = (unsigned char)nlead;
        __syncthreads();
        // the tile's earlier chunks, and this chunk's earlier waves
        if (valid) {
            unsigned n = (unsigned)hist[b];
#pragma unroll
            for (int k = 0; k < NW / 4; ++k) {
                const int w = wave - 4 * k;   // earlier waves in this word
                const unsigned v = whist[b * (NW / 4) + k];
                if (w >= 4) n = __builtin_amdgcn_sad_u8(v, 0u, n);
                else if (w > 0) n = __builtin_amdgcn_sad_u8(v & ((1u << (8 * w)) - 1u), 0u, n);
            }
            rk += (int)n;
        }
        __syncthreads();
        if (lead) {
            atomicAdd(&hist[b], nlead);
            reinterpret_cast<unsigned char *>(whist)[NW * b + wave] = 0;
        }
        if (MODE == 0 && valid) {
            bin[i] = S * NBINS + b;
            rank[i] = rk;
        }
        if (MODE == 2 && valid) {
            const int64_t d = (int64_t)off_new[dcell] + cnt[(size_t)S * NBINS + b] + rk;
            if (d >= 0 && d < np) {
                o.x[d] = ox_;
                o.y[d] = oy_;
                o.px[d] = opx;
                o.py[d] = opy;
                o.pz[d] = opz;
                o.p6[d] = p6;
                o.p7[d] = p7;
                if (!uq) o.q[d] = q;   // a uniform q is already in place
            } else {
                atomicMax(err, 1 << 29);   // the two passes disagree: never expected
            }
        }
    }
    if (MODE == 2) {
        if (tid == 0) tot[S] = 0;
        return;
    }
    __syncthreads();
    __shared__ int s_tot[9];   // particles bound for each neighbour
    if (MODE == 1 && tid < 9) s_tot[tid] = 0;
    for (int n = tid; n < NBINS; n += NT) cnt[(size_t)S * NBINS + n] = hist[n];
    if (MODE != 1) return;
    __syncthreads();
    for (int n = tid; n < NBINS; n += NT) {   // a wave's bins are one neighbour's
        int h = hist[n];
        if (!__any(h)) continue;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) h += __shfl_xor(h, o);
        if (lane == 0) atomicAdd(&s_tot[n / TCELLS], h);
    }
    __syncthreads();
    if (tid < 9 && s_tot[tid])
        atomicAdd(&tot[wrap1(ty0 + tid / 3 - 1, g.my1) * g.mx1 + wrap1(tx0 + tid % 3 - 1, g.mx1)],
                  s_tot[tid]);
}

// Per destination cell d (in tile T, local cell cl): its particles come from
// bins (T - dir(nb), nb, cl), nb = 0..8.  Taken in nb order, the bin counts
// are turned into each bin's start within the cell, and the cell count is
// written for the scan; count[ncells] = 0.
__global__ void k_bin_starts(TileGeom g, int *cnt, int *count)
{
    const int d = blockIdx.x * blockDim.x + threadIdx.x;
    const int ncells = g.mx1 * g.my1 * TCELLS;
    if (d == ncells) count[d] = 0;
    if (d >= ncells) return;
    const int T = d >> 8, cl = d & 255;
    const int tx = T % g.mx1, ty = T / g.mx1;
    int run = 0;
    for (int nb = 0; nb < 9; ++nb) {
        const int dirx = nb % 3 - 1, diry = nb / 3 - 1;
        const int sx = wrap1(tx - dirx, g.mx1), sy = wrap1(ty - diry, g.my1);
        const size_t k = (size_t)(sy * g.mx1 + sx) * NBINS + nb * TCELLS + cl;
        const int c = cnt[k];
        cnt[k] = run;
        run += c;
    }
    count[d] = run;
}

// Totals of groups of GROUP tiles, for k_bin_offsets on large grids
__global__ void __launch_bounds__(GROUP) k_group_totals(int ntiles, const int *tot, int *grp)
{
    __shared__ int s[GROUP / 64];
    const int t = blockIdx.x * GROUP + threadIdx.x;
    int v = t < ntiles ? tot[t] : 0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        int sum = 0;
        for (int w = 0; w < GROUP / 64; ++w) sum += s[w];
        grp[blockIdx.x] = sum;
    }
}

// The same as k_bin_starts, and the new cell offsets in place of the counts: a
// tile's first particle is the sum of the tiles before it, from the totals that
// the counting push has added up (integer sums: any order), and its cells
// follow by a prefix sum over the workgroup.  grp (above 8192 tiles): the
// totals of the groups of tiles before; below, reading at most 32 KB of totals
// per workgroup from L2 costs less than the launch that makes them.  One launch
// for three of the counts' kernel and a library scan: 27 us at 1024^2 (4.6 of
// them the scan's set-up) become 16, and 10 become 3.4 at 128^2.
__global__ void __launch_bounds__(TCELLS)
k_bin_offsets(TileGeom g, int *cnt, const int *__restrict__ tot, const int *__restrict__ grp,
              int *off)
{
    __shared__ int s_sum[2][TCELLS / 64];
    const int T = blockIdx.x, cl = threadIdx.x, lane = cl & 63, wave = cl >> 6;
    const int ntiles = g.mx1 * g.my1;
    const int tx = T % g.mx1, ty = T / g.mx1;
    size_t k[9];
    int c[9];
#pragma unroll
    for (int nb = 0; nb < 9; ++nb) {
        const int sx = wrap1(tx - (nb % 3 - 1), g.mx1), sy = wrap1(ty - (nb / 3 - 1), g.my1);
        k[nb] = (size_t)(sy * g.mx1 + sx) * NBINS + nb * TCELLS + cl;
        c[nb] = cnt[k[nb]];
    }
    int base = 0;
    int t0 = 0;
    if (grp) {
        t0 = T / GROUP * GROUP;
        for (int i = cl; i < T / GROUP; i += TCELLS) base += grp[i];
    }
    for (int i = t0 + cl; i < T; i += TCELLS) base += tot[i];
    int run = 0;
#pragma unroll
    for (int nb = 0; nb < 9; ++nb) {
        cnt[k[nb]] = run;
        run += c[nb];
    }
    int pre = run;   // inclusive prefix over the wave
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(pre, o);
        if (lane >= o) pre += v;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) base += __shfl_xor(base, o);
    if (lane == 63) {
        s_sum[0][wave] = pre;
        s_sum[1][wave] = base;
    }
    __syncthreads();
    int first = 0;
#pragma unroll
    for (int w = 0; w < TCELLS / 64; ++w) first += s_sum[1][w] + (w < wave ? s_sum[0][w] : 0);
    off[T * TCELLS + cl] = first + pre - run;
    if (T == ntiles - 1 && cl == TCELLS - 1) off[ntiles * TCELLS] = first + pre;
}

// destination of particle i: off[cell] + start of its bin in the cell + rank
template <typename R>
__global__ void k_scatter(int64_t np, Soa<R> a, Soa<R> b, const int *bin, const int *rank,
                          const int *cnt, const int *off, int mx1, int my1)
{
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= np) return;
    // the record is read completely, and first, before any store (the
    // compiler may not move a load of a past a store to b, which it cannot
    // prove disjoint); its loads overlap those of the destination
    const R v0 = a.x[i], v1 = a.y[i], v2 = a.px[i], v3 = a.py[i], v4 = a.pz[i], v5 = a.p6[i],
            v6 = a.p7[i], v7 = a.q[i];
    __builtin_amdgcn_sched_barrier(0);   // keep these loads ahead of the lookups
    const int bi = bin[i], rk = rank[i];
    const int S = bi / NBINS, bb = bi - S * NBINS, nb = bb >> 8, cl = bb & 255;
    const int tx = wrap1(S % mx1 + nb % 3 - 1, mx1), ty = wrap1(S / mx1 + nb / 3 - 1, my1);
    const int d = off[(ty * mx1 + tx) * TCELLS + cl] + cnt[bi] + rk;
    b.x[d] = v0;
    b.y[d] = v1;
    b.px[d] = v2;
    b.py[d] = v3;
    b.pz[d] = v4;
    b.p6[d] = v5;
    b.p7[d] = v6;
    b.q[d] = v7;
}

// cell keys of unsorted particles (initial load and uploads), with their
// index for a stable sort and a per-cell count
template <typename R>
__global__ void k_keys(int64_t np, const R *x, const R *y, int nx, int ny, int mx1, int *key,
                       int *idx, int *count, int *err)
{
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= np) return;
    R xv = x[i], yv = y[i];
    int cx = (int)xv, cy = (int)yv;
    if (!(xv >= R(0) && yv >= R(0) && cx < nx && cy < ny)) {
        atomicMax(err, 1 << 30);
        cx = min(max(cx, 0), nx - 1);
        cy = min(max(cy, 0), ny - 1);
    }
    int k = cell_key(cx, cy, mx1);
    key[i] = k;
    idx[i] = (int)i;
    atomicAdd(&count[k], 1);
}

// the same for keys computed on the host (FP32 tile-relative records)
__global__ void k_count_keys(int64_t np, const int *key, int *idx, int *count)
{
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= np) return;
    idx[i] = (int)i;
    atomicAdd(&count[key[i]], 1);
}

// b[p] = a[src[p]]
template <typename R>
__global__ void k_gather(int64_t np, Soa<R> a, Soa<R> b, const int *src)
{
    int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (p >= np) return;
    const int i = src[p];
    const R v0 = a.x[i], v1 = a.y[i], v2 = a.px[i], v3 = a.py[i], v4 = a.pz[i], v5 = a.p6[i],
            v6 = a.p7[i], v7 = a.q[i];
    b.x[p] = v0;
    b.y[p] = v1;
    b.px[p] = v2;
    b.py[p] = v3;
    b.pz[p] = v4;
    b.p6[p] = v5;
    b.p7[p] = v6;
    b.q[p] = v7;
}

// the move-check word into pinned host memory, in stream order (a kernel
// store instead of a copy-engine transfer between the slice's kernels):
// h_err[0] = the word; h_err[1] = the slice of the first post that saw it
// set (the word stays set until the host clears it, so that is the slice
// whose push set it)
__global__ void k_post_err(const int *err, int *h_err, int slice)
{
    if (threadIdx.x == 0) {
        const int e = *err;
        h_err[0] = e;
        if (e && h_err[1] == 0) h_err[1] = slice;
        __threadfence_system();
    }
}

__global__ void k_zero_int(int *p, int n)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0;
}

static TileGeom geom(qp_ctx *c) { return TileGeom{c->nx, c->ny, c->mx1, c->my1, c->ldr}; }

static dim3 pgrid(int64_t n) { return dim3((unsigned)((n + 255) / 256)); }

// cell offsets from the per-cell counts
static int scan_counts(qp_species *sp)
{
    qp_ctx *c = sp->ctx;
    size_t tb = sp->scan_bytes;
    QP_HIP(hipcub::DeviceScan::ExclusiveSum(sp->scan_tmp.p, tb, sp->count.as<int>(),
                                            sp->off.as<int>(), c->ncells + 1,
                                            c->stream));
    return QP_OK;
}

static int zero_counts(qp_species *sp)
{
    qp_ctx *c = sp->ctx;
    hipLaunchKernelGGL(k_zero_int, dim3(1024), dim3(256), 0, c->stream, sp->count.as<int>(),
                       c->ncells + 1);
    QP_LAUNCH_CHECK();
    return QP_OK;
}

static int check_err(qp_species *sp, const char *what)
{
    qp_ctx *c = sp->ctx;
    int h = 0;
    QP_HIP(hipMemcpyAsync(&h, sp->err.p, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    QP_HIP(hipStreamSynchronize(c->stream));
    if (h) {
        QP_HIP(hipMemsetAsync(sp->err.p, 0, sizeof(int), c->stream));
        if (h >= (1 << 30)) set_error("%s: particle position outside the grid", what);
        else if (h >= (1 << 29)) set_error("%s: the push's two passes disagree", what);
        else set_error("%s: particle left its tile by more than one tile (tile %d)", what, h);
        return QP_ERR_CHECK;
    }
    return QP_OK;
}

// sort an arbitrary particle order by cell: keys, a stable radix sort of
// (key, index), offsets, then a gather into the alternate arrays.  hkeys:
// the cell keys, computed on the host (FP32 records hold tile-relative
// positions, from which the device cannot tell the tile)
template <typename R>
static int rebin_unsorted(qp_species *sp, const std::vector<int> *hkeys = nullptr)
{
    qp_ctx *c = sp->ctx;
    int rc = zero_counts(sp);
    if (rc) return rc;
    const int64_t np = sp->np;
    DevBuf keys2, idx2, tmp;
    rc = keys2.alloc((size_t)np * 4 + 4);
    if (!rc) rc = idx2.alloc((size_t)np * 4 + 4);
    if (rc) return rc;
    size_t tb = 0;
    int bits = 1;
    while ((1 << bits) < c->ncells) ++bits;
    QP_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, sp->key.as<int>(), keys2.as<int>(),
                                              sp->slot.as<int>(), idx2.as<int>(), (int)np, 0,
                                              bits, c->stream));
    rc = tmp.alloc(tb + 256);
    if (rc) return rc;
    if (hkeys) {
        QP_REQUIRE((int64_t)hkeys->size() == np, QP_ERR_ARG, "particle load: %zu keys for %lld",
                   hkeys->size(), (long long)np);
        QP_HIP(hipMemcpyAsync(sp->key.p, hkeys->data(), (size_t)np * sizeof(int),
                              hipMemcpyHostToDevice, c->stream));
        hipLaunchKernelGGL(k_count_keys, pgrid(np), dim3(256), 0, c->stream, np,
                           sp->key.as<const int>(), sp->slot.as<int>(), sp->count.as<int>());
    } else {
        ProfScope _ps(c, QP_PROF_SORT, 2.0 * sizeof(R) * (double)np);
        hipLaunchKernelGGL(k_keys<R>, pgrid(np), dim3(256), 0, c->stream, np, sp->a[0].as<R>(),
                           sp->a[1].as<R>(), c->nx, c->ny, c->mx1, sp->key.as<int>(),
                           sp->slot.as<int>(), sp->count.as<int>(), sp->err.as<int>());
    }
    QP_LAUNCH_CHECK();
    QP_HIP(hipcub::DeviceRadixSort::SortPairs(tmp.p, tb, sp->key.as<int>(), keys2.as<int>(),
                                              sp->slot.as<int>(), idx2.as<int>(), (int)np, 0,
                                              bits, c->stream));
    rc = scan_counts(sp);
    if (rc) return rc;
    hipLaunchKernelGGL(k_gather<R>, pgrid(np), dim3(256), 0, c->stream, np, soa<R>(sp->a),
                       soa<R>(sp->b), idx2.as<const int>());
    QP_LAUNCH_CHECK();
    for (int k = 0; k < 8; ++k) std::swap(sp->a[k], sp->b[k]);
    QP_HIP(hipStreamSynchronize(c->stream));   // the temporaries are freed on return
    return check_err(sp, "particle load");
}

template <typename R>
static int deposit_border(qp_ctx *c, const DepOut<R> &out, int ncomp, int fold,
                          const R *halo = nullptr, int bands = 1, BorderJob *job = nullptr)
{
    QP_REQUIRE(ncomp >= 1 && ncomp <= 8, QP_ERR_ARG, "deposit border: %d components", ncomp);
    TileGeom g = geom(c);
    const int rb = TILE / bands, myb = c->my1 * bands;
    if (job) {
        *job = BorderJob{};
        job->halo = halo ? halo : c->halo.as<R>();
        job->rb = rb;
        job->fold = fold;
        job->n = ncomp;
        for (int k = 0; k < ncomp; ++k) {
            job->p[k] = out.p[k];
            job->inner[k] = out.inner[k];
            job->outer[k] = out.outer[k];
            job->p2[k] = out.p2[k];
        }
        job->scale = (double)out.scale;
        job->scale2 = (double)out.scale2;
        return QP_OK;
    }
    int n = (myb + 1) * (c->nx + 1) + (c->mx1 + 1) * myb * (rb - 1);
    {
    ProfScope _ps(c, QP_PROF_BORDER, 2.0 * ncomp * (double)n * sizeof(R));
    auto kern = bands == 4 ? k_deposit_border<R, TILE / 4>
              : bands == 2 ? k_deposit_border<R, TILE / 2> : k_deposit_border<R, TILE>;
    hipLaunchKernelGGL(kern, dim3((n + 255) / 256, ncomp), dim3(256), 0, c->stream,
                       g, halo ? halo : c->halo.as<R>(),
                       (size_t)c->ntiles * bands * band_halo(rb), out, fold, c->skip);
    }
    QP_LAUNCH_CHECK();
    return QP_OK;
}

// Deposit launch shapes: rows per group RG (16/RG lanes per cell; 0: chosen
// per tile), staging chunk CH and a waves-per-SIMD floor WPE (4 caps the
// kernel at 128 VGPRs).  Variant 0 of each table is the default; qp_ctx_tune
// selects another.  The FP32 current deposit's default chooses its rows per
// group per tile, keeping a group within two staging chunks (THR = 8):
// 472.4-472.5 slices/s on whole 1024^2, 16 ppc steps at nb/n0 = 10, against
// 464.0 within 1.5 chunks (variant 12), 455.0 within one (variant 14) and
// 434.8-437.2 with a fixed RG = 8 (variant 11); FP64 likewise, 242.9-243.4
// against 233.9-234.3 with a fixed RG = 8 (variant 11).
struct DepShape {
    int rg, ch, wpe;
    int wave;          // current deposit: 1 k_amjdp_w (independent waves, staging
                       // chunk ch per wave); 2 k_amjdp_pf (next chunk prefetched
                       // into registers); 3 k_amjdp_dma (FP32: chunks copied into
                       // LDS by LDS-DMA, double-buffered)
    int thr = 4;       // rg = 0: a group's share of the tile's particles is kept
                       // at or below thr/4 of the chunk
};
template <typename R> struct DepTab;
template <> struct DepTab<float> {
    static constexpr DepShape q[] = {{16, 4096, 1, 0}, {16, 1024, 1, 0}, {8, 2048, 1, 0},
                                     {16, 2048, 1, 0}};
    static constexpr DepShape j[] = {{0, 1024, 4, 0, 8}, {8, 1024, 1, 0}, {4, 1024, 4, 0},
                                     {16, 1024, 4, 0}, {4, 512, 4, 0},  {8, 512, 1, 0},
                                     {2, 256, 1, 1},   {2, 128, 1, 1},  {8, 1024, 1, 2},
                                     {8, 512, 1, 2},   {8, 512, 1, 3},  {8, 1024, 4, 0},
                                     {0, 1024, 4, 0, 6}, {0, 1024, 4, 0, 10}, {0, 1024, 4, 0, 4}};
};
template <> struct DepTab<double> {
    static constexpr DepShape q[] = {{8, 1024, 1, 0}, {8, 2048, 1, 0}, {16, 1024, 1, 0},
                                     {8, 512, 1, 0}};
    static constexpr DepShape j[] = {{0, 1024, 1, 0, 8}, {4, 1024, 1, 0}, {4, 512, 1, 0},
                                     {8, 512, 1, 0},  {2, 512, 1, 0},  {16, 512, 1, 0},
                                     {2, 128, 1, 1},  {2, 64, 1, 1},   {8, 512, 1, 2},
                                     {8, 256, 1, 2},   {8, 256, 1, 0},  {8, 1024, 1, 0},
                                     {0, 1024, 1, 0, 6}, {0, 1024, 1, 0, 10}, {0, 1024, 1, 0, 4}};
};

// kernels using more than 64 KB of dynamic LDS ask for it once
template <typename K>
static int allow_lds(K kernel, size_t bytes, qp_ctx *c)
{
    QP_REQUIRE(bytes <= c->max_lds, QP_ERR_UNSUPPORTED, "kernel needs %zu B of LDS (limit %zu)",
               bytes, c->max_lds);
    if (bytes > 65536)
        QP_HIP(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)bytes));
    return QP_OK;
}

template <typename R, int V>
static int deposit_q_v(qp_species *sp, const DepOut<R> &out, R *halo, const BeamPlane *bp)
{
    qp_ctx *c = sp->ctx;
    constexpr DepShape d = DepTab<R>::q[V];
    const size_t lds = ((sp->q_uniform ? 2 : 3) * (size_t)Stage<d.ch>::N + 289) * sizeof(R);
    auto kern = sp->q_uniform ? k_deposit_q<R, d.rg, d.ch, d.wpe, true>
                              : k_deposit_q<R, d.rg, d.ch, d.wpe, false>;
    int rc = allow_lds(kern, lds, c);
    if (rc) return rc;
    {
    // x, y (and q unless uniform) per particle, one plane
    const double words = sp->q_uniform ? 2.0 : 3.0;
    ProfScope _ps(c, QP_PROF_DEPOSIT_Q, (words * sp->np + (c->nx + 1.0) * (c->ny + 1.0)) * sizeof(R));
    hipLaunchKernelGGL(kern, dim3(c->ntiles + (bp ? BEAM_BLOCKS : 0)), dim3(256), lds, c->stream,
                       geom(c), soa<R>(sp->a), sp->off.as<int>(), out, halo, (R)sp->q_value,
                       bp ? *bp : BeamPlane{});
    }
    QP_LAUNCH_CHECK();
    return QP_OK;
}

// halo: the tile-border buffer (null: the context's)
template <typename R>
static int deposit_q_out(qp_species *sp, const DepOut<R> &out, R *halo = nullptr,
                         const BeamPlane *bp = nullptr, BorderJob *job = nullptr)
{
    int rc;
    if (!halo) halo = sp->ctx->halo.as<R>();
    switch (sp->ctx->tune[QP_TUNE_DEPOSIT_Q]) {
    case 1: rc = deposit_q_v<R, 1>(sp, out, halo, bp); break;
    case 2: rc = deposit_q_v<R, 2>(sp, out, halo, bp); break;
    case 3: rc = deposit_q_v<R, 3>(sp, out, halo, bp); break;
    default: rc = deposit_q_v<R, 0>(sp, out, halo, bp); break;
    }
    if (rc) return rc;
    return deposit_border<R>(sp->ctx, out, 1, 1, halo, 1, job);
}

// species charge into a real-space plane (overwritten), guard-folded
template <typename R> static int deposit_q_t(qp_species *sp, R *plane)
{
    return deposit_q_out<R>(sp, dep_plain<R>(&plane, 1));
}

// Marks the species' charge uniform (or not); a uniform q is written into
// both particle buffers, so no permutation has to move it
static int set_q_uniform(qp_species *sp, bool uniform, double v)
{
    sp->q_uniform = uniform;
    sp->q_value = v;
    if (!uniform || sp->np == 0) return QP_OK;
    int rc = launch_fill(sp->ctx, sp->a[7].p, (size_t)sp->np, v);
    if (!rc) rc = launch_fill(sp->ctx, sp->b[7].p, (size_t)sp->np, v);
    return rc;
}

// The quiet-start lattice of dist2d_000 (fdist2d_class.f03:212-316), one
// rank: x = (ix + 0.5)/xppc + i - 1, i = 2..nx-1, and y likewise over j =
// 2..ny, each particle of charge qm; with a transverse profile its points are
// weighted or dropped.  Lengths in grid units.
struct Lattice {
    int nx, ny, mx1, xppc, yppc, profile, nr;
    double qm, cx, cy, irx, iry, orx, ory, r0, sigr;
    const double *r, *fr;   // 12: the radial points
};

// The transverse profile at a lattice point (x, y): false drops it; w is its
// charge weight.  In the reference's operation order, without contraction:
//   10 (dist2d_010, fdist2d_class.f03:438-441): dropped inside the inner or
//      outside the outer ellipse;
//   11 (dist2d_011, :633-645): w = exp(-(r - r0)^2 * 0.5 / sigr^2);
//   12 (dist2d_012, :836-856): dropped outside [r(1), r(n)], else w = fr
//      interpolated linearly at r; a pair of points that does not increase,
//      met on the way to r, sets *bad.
__device__ bool lattice_weight(const Lattice &L, double x, double y, double &w, int *bad)
{
#pragma clang fp contract(off)
    w = 1.0;
    if (L.profile == 0) return true;
    if (L.profile == 10) {
        const double iirx2 = 1.0 / (L.irx * L.irx), iiry2 = 1.0 / (L.iry * L.iry);
        const double iorx2 = 1.0 / (L.orx * L.orx), iory2 = 1.0 / (L.ory * L.ory);
        const double ddx = (x - L.cx) * (x - L.cx), ddy = (y - L.cy) * (y - L.cy);
        return !((ddx * iirx2 + ddy * iiry2 < 1.0) || (ddx * iorx2 + ddy * iory2 > 1.0));
    }
    const double rr = sqrt((x - L.cx) * (x - L.cx) + (y - L.cy) * (y - L.cy));
    if (L.profile == 11) {
        const double isigr2 = 0.5 / (L.sigr * L.sigr);
        w = exp(-((rr - L.r0) * (rr - L.r0)) * isigr2);
        return true;
    }
    if (rr < L.r[0] || rr > L.r[L.nr - 1]) return false;
    for (int i = 1; i < L.nr; ++i) {
        const double ra = L.r[i - 1], rb = L.r[i];
        if (rb <= ra) {
            *bad = 1;
            return false;
        }
        if (rr <= rb) {
            w = L.fr[i - 1] + (L.fr[i] - L.fr[i - 1]) / (rb - ra) * (rr - ra);
            break;
        }
    }
    return true;
}

// the cell of sort key k, and whether the lattice covers it
__device__ __forceinline__ bool lattice_cell(const Lattice &L, int k, int &cx, int &cy)
{
    const int t = k / TCELLS, l = k % TCELLS;
    cx = (t % L.mx1) * TILE + (l & 15);
    cy = (t / L.mx1) * TILE + (l >> 4);
    return cx >= 1 && cx <= L.nx - 2 && cy >= 1 && cy <= L.ny - 1;
}

__device__ __forceinline__ double lattice_at(int i, int n, int cell)
{
#pragma clang fp contract(off)
    return (i + 0.5) / n + (cell + 1) - 1;
}

// particles of every cell (and count[ncells] = 0), for the scan
__global__ void __launch_bounds__(256) k_load_count(Lattice L, int ncells, int *count, int *bad)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k > ncells) return;
    int cx, cy, n = 0, b = 0;
    if (k < ncells && lattice_cell(L, k, cx, cy)) {
        if (L.profile == 0 || L.profile == 11) n = L.xppc * L.yppc;
        else
            for (int ix = 0; ix < L.xppc; ++ix)
                for (int iy = 0; iy < L.yppc; ++iy) {
                    double w;
                    if (lattice_weight(L, lattice_at(ix, L.xppc, cx), lattice_at(iy, L.yppc, cy),
                                       w, &b))
                        ++n;
                }
    }
    count[k] = n;
    if (b) *bad = 1;
}

// The loaded particles at their sorted places, one workgroup per tile.  Bound
// by its stores: all 8 words of a particle are written once and nothing is
// read but the offsets.  The lattice is computed where it is stored, so no
// host array, copy or sort takes part: a reload of 1024 x 1024 cells, 16
// particles each, in FP32 took 72 ms with a host loop, its copies and a radix
// sort, and takes 0.20 ms here (FP64: 0.36 ms).
// Without dropped points every covered cell of the tile holds the same count
// and the cells form a rectangle, so thread by thread the particles are taken
// in their sorted order and the stores are coalesced (one thread per cell took
// 1.74 ms for that reload).  DROP: one thread per cell keeps the order of the
// kept points.  q2: the alternate buffer's charges, filled too when all are
// equal (null with a weighted profile).
template <typename R>
__device__ __forceinline__ void load_one(const Lattice &L, int ix, int iy, int cx, int cy, int &p,
                                         const Soa<R> &s, R *q2, R p67)
{
    int bad = 0;
    const double x = lattice_at(ix, L.xppc, cx), y = lattice_at(iy, L.yppc, cy);
    const int x0 = TileRel<R>::on ? cx & ~(TILE - 1) : 0, y0 = TileRel<R>::on ? cy & ~(TILE - 1) : 0;
    double w;
    if (!lattice_weight(L, x, y, w, &bad)) return;
    const R q = (R)(L.qm * w);
    s.x[p] = (R)(x - (double)x0);
    s.y[p] = (R)(y - (double)y0);
    s.px[p] = R(0);
    s.py[p] = R(0);
    s.pz[p] = R(0);
    s.p6[p] = p67;
    s.p7[p] = p67;
    s.q[p] = q;
    if (q2) q2[p] = q;
    ++p;
}

template <typename R, bool DROP>
__global__ void __launch_bounds__(256)
k_load_fill(Lattice L, const int *__restrict__ off, Soa<R> s, R *q2, R p67)
{
    const int tile = blockIdx.x, kb = tile * TCELLS;
    if (DROP) {
        int cx, cy;
        if (!lattice_cell(L, kb + threadIdx.x, cx, cy)) return;
        int p = off[kb + threadIdx.x];
        for (int ix = 0; ix < L.xppc; ++ix)
            for (int iy = 0; iy < L.yppc; ++iy) load_one(L, ix, iy, cx, cy, p, s, q2, p67);
        return;
    }
    const int x0 = (tile % L.mx1) * TILE, y0 = (tile / L.mx1) * TILE;
    const int xa = max(x0, 1), ya = max(y0, 1);
    const int w = min(x0 + TILE - 1, L.nx - 2) - xa + 1;   // covered columns of the tile
    const int ppc = L.xppc * L.yppc, p0 = off[kb], n = off[kb + TCELLS] - p0;
    for (int i = threadIdx.x; i < n; i += TCELLS) {
        const int cell = i / ppc, m = i - cell * ppc, ix = m / L.yppc;
        int p = p0 + i;
        load_one(L, ix, m - ix * L.yppc, xa + cell % w, ya + cell / w, p, s, q2, p67);
    }
}

// (re)load of the plasma, in cell order
template <typename R>
static int distribute(qp_species *sp)
{
    qp_ctx *c = sp->ctx;
    const int xppc = sp->p.ppc[0], yppc = sp->p.ppc[1];
    const bool weighted = sp->profile == 11 || sp->profile == 12;
    const bool drops = sp->profile == 10 || sp->profile == 12;
    Lattice L{};
    L.nx = c->nx; L.ny = c->ny; L.mx1 = c->mx1; L.xppc = xppc; L.yppc = yppc;
    L.profile = sp->profile;
    L.qm = sp->den_factor * sp->p.density * sp->p.q / std::fabs(sp->p.q) / (double)xppc /
           (double)yppc;
    L.cx = sp->pcx; L.cy = sp->pcy;
    L.irx = sp->irx; L.iry = sp->iry; L.orx = sp->orx; L.ory = sp->ory;
    L.r0 = sp->r0; L.sigr = sp->sigr;
    L.nr = (int)sp->pr.size();
    if (L.nr) {
        QP_REQUIRE(sp->radial.bytes >= 2 * L.nr * sizeof(double), QP_ERR_STATE,
                   "plasma load: no radial points");
        L.r = sp->radial.as<double>();
        L.fr = L.r + L.nr;
    }
    // the flag of a bad radial point: a word of the (unused) index array
    int *bad = sp->slot.as<int>();
    const dim3 grid((c->ncells + 256) / 256);
    int64_t n = (int64_t)(c->nx - 2) * (c->ny - 1) * xppc * yppc;
    if (drops) {
        hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(64), 0, c->stream, bad, 1);
        QP_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(k_load_count, grid, dim3(256), 0, c->stream, L, c->ncells,
                       sp->count.as<int>(), bad);
    QP_LAUNCH_CHECK();
    if (drops) {
        int h = 0;
        QP_HIP(hipMemcpyAsync(&h, bad, sizeof(int), hipMemcpyDeviceToHost, c->stream));
        QP_HIP(hipStreamSynchronize(c->stream));
        QP_REQUIRE(!h, QP_ERR_ARG, "dist2d_012: r is not monotonically increasing!");
    }
    int rc = scan_counts(sp);
    if (rc) return rc;
    if (drops) {
        int h = 0;
        QP_HIP(hipMemcpyAsync(&h, sp->off.as<int>() + c->ncells, sizeof(int),
                              hipMemcpyDeviceToHost, c->stream));
        QP_HIP(hipStreamSynchronize(c->stream));
        n = h;
    }
    sp->np = n;
    // p6 = p7 = 1 at rest (0 in the FP32 deviation form)
    const R p67 = P67Dev<R>::on ? R(0) : R(1);
    auto fill = drops ? k_load_fill<R, true> : k_load_fill<R, false>;
    hipLaunchKernelGGL(fill, dim3(c->ntiles), dim3(256), 0, c->stream, L,
                       sp->off.as<const int>(), soa<R>(sp->a),
                       weighted ? nullptr : sp->b[7].as<R>(), p67);
    QP_LAUNCH_CHECK();
    sp->q_uniform = !weighted;
    sp->q_value = L.qm;
    return check_err(sp, "particle load");
}

// The density factor at propagation distance s of dist2d_000
// (fdist2d_class.f03:233-251): 1 for a uniform plasma; else the linear
// interpolation of fs between the points s(i-1) <= s <= s(i), with the
// reference's checks (s inside the points; the points increasing up to the
// segment found)
static int den_factor_at(qp_species *sp, double s)
{
    sp->den_factor = 1.0;
    const size_t n = sp->lp_s.size();
    if (n == 0) return QP_OK;
    const std::vector<double> &ps = sp->lp_s, &fs = sp->lp_fs;
    QP_REQUIRE(!(s < ps[0] || s > ps[n - 1]), QP_ERR_ARG,
               "dist2d_000: The s is out of the bound! (s = %g)", s);
    for (size_t i = 1; i < n; ++i) {
        QP_REQUIRE(!(ps[i] < ps[i - 1]), QP_ERR_ARG,
                   "dist2d_000: s is not monotonically increasing!");
        if (s <= ps[i]) {
            sp->den_factor = fs[i - 1] + (fs[i] - fs[i - 1]) / (ps[i] - ps[i - 1]) * (s - ps[i - 1]);
            break;
        }
    }
    return QP_OK;
}

// renew: particles and qn = -(folded deposit of the fresh plasma)
template <typename R>
static int renew_t(qp_species *sp)
{
    int rc = distribute<R>(sp);
    if (rc) return rc;
    rc = deposit_q_t<R>(sp, sp->qn->rs.as<R>());
    if (rc) return rc;
    sp->qn->state = 0;
    double m1 = -1.0;
    return qp_field2d_mult(sp->qn, sp->qn, 0, nullptr, nullptr, &m1);
}

template <typename R>
static int alloc_particles(qp_species *sp, int64_t np)
{
    qp_ctx *c = sp->ctx;
    for (int k = 0; k < 8; ++k) {
        int rc = sp->a[k].alloc((size_t)np * sizeof(R));
        if (!rc) rc = sp->b[k].alloc((size_t)np * sizeof(R));
        if (rc) return rc;
    }
    int rc = sp->key.alloc((size_t)np * 4);
    if (!rc) rc = sp->slot.alloc((size_t)np * 4);
    if (!rc) rc = sp->count.alloc((size_t)(c->ncells + 1) * 4);
    if (!rc) rc = sp->bins.alloc((size_t)c->ntiles * NBINS * 4);
    if (!rc) rc = sp->tot.alloc((size_t)(c->ntiles + (c->ntiles + GROUP - 1) / GROUP) * 4);
    if (!rc) rc = sp->off.alloc((size_t)(c->ncells + 1) * 4);
    if (!rc) rc = sp->off_new.alloc((size_t)(c->ncells + 1) * 4);
    if (!rc) rc = sp->err.alloc(sizeof(int));
    if (rc) return rc;
    QP_HIP(hipHostMalloc((void **)&sp->h_err, 2 * sizeof(int), hipHostMallocDefault));
    sp->h_err[0] = sp->h_err[1] = 0;
    QP_HIP(hipEventCreateWithFlags(&sp->err_ev, hipEventDisableTiming));
    sp->scan_bytes = 0;
    QP_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, sp->scan_bytes, sp->count.as<int>(),
                                            sp->off.as<int>(), c->ncells + 1, c->stream));
    return sp->scan_tmp.alloc(sp->scan_bytes + 256);
}

template <typename R>
static int extpsi_t(qp_species *sp, const qp_field2d *psi, double dex)
{
    qp_ctx *c = sp->ctx;
    if (sp->np == 0) return QP_OK;
    {
    ProfScope _ps(c, QP_PROF_EXTPSI, (6.0 * sp->np + (c->nx + 1.0) * (c->ny + 1.0)) * sizeof(R));
    hipLaunchKernelGGL(k_extpsi<R>, pgrid(sp->np), dim3(256), 0, c->stream, sp->np, c->nx, c->ny,
                       c->ldr, soa<R>(sp->a), psi->rs.as<R>(), (R)sp->qbm, (R)dex,
                       sp->off.as<int>(), c->mx1, c->ntiles);
    }
    QP_LAUNCH_CHECK();
    return QP_OK;
}

template <typename R, int V, int B = 1, bool ADD = false>
static int amjdp_v(qp_species *sp, const qp_field2d *ef, const qp_field2d *bf,
                   const qp_field2d *psit, double dex, const DepOut<R> &out,
                   const qp_field2d *psi)
{
    qp_ctx *c = sp->ctx;
    const size_t pl = c->rplane;
    const size_t hcs = (size_t)c->ntiles * B * band_halo(TILE / B);
    constexpr DepShape d = DepTab<R>::j[V];
    size_t lds;
    void (*kern)(TileGeom, Soa<R>, const int *, const R *, const R *, const R *, size_t,
                 DepOut<R>, R *, size_t, R, R, R, const int *, const R *, R);
    if constexpr (d.wave == 1) {
        lds = (4 * 7 * (size_t)Stage<d.ch>::N + 8 * 8 * 51) * sizeof(R);
        kern = k_amjdp_w<R, d.ch>;
    } else if constexpr (d.wave == 2) {
        lds = (7 * (size_t)Stage<d.ch>::N + 8 * 289) * sizeof(R);
        kern = k_amjdp_pf<R, d.rg, d.ch>;
    } else if constexpr (d.wave == 3) {
        static_assert(std::is_same<R, float>::value, "LDS-DMA staging is FP32 only");
        lds = (2 * 7 * (size_t)(d.ch + d.ch / 64) + 8 * 289) * sizeof(R);
        kern = k_amjdp_dma<d.rg, d.ch>;
    } else {
        lds = (7 * (size_t)Stage<d.ch>::N + 8 * 289) * sizeof(R);
        if (sp->q_uniform)
            kern = psi ? k_amjdp<R, d.rg, d.ch, d.wpe, true, true, d.thr, B, ADD>
                       : k_amjdp<R, d.rg, d.ch, d.wpe, false, true, d.thr, B, ADD>;
        else
            kern = psi ? k_amjdp<R, d.rg, d.ch, d.wpe, true, false, d.thr, B, ADD>
                       : k_amjdp<R, d.rg, d.ch, d.wpe, false, false, d.thr, B, ADD>;
    }
    int rc = allow_lds(kern, lds, c);
    if (rc) return rc;
    {
    // with psi: p6 and p7 written but, by the default form, not read, and one more
    // plane; a uniform q is not read (by the kernels with a uniform-charge form)
    const double words = (psi ? (d.wave == 0 ? 7.0 : 9.0) : 8.0) - (sp->q_uniform && d.wave == 0 ? 1.0 : 0.0);
    const double planes = psi ? 15.0 : 14.0;
    ProfScope _ps(c, QP_PROF_AMJDP, (words * sp->np + planes * (c->nx + 1.0) * (c->ny + 1.0)) * sizeof(R));
    hipLaunchKernelGGL(kern, dim3(c->ntiles * B), dim3(256), lds, c->stream, geom(c),
                       soa<R>(sp->a), sp->off.as<int>(), ef->rs.as<R>(), bf->rs.as<R>(),
                       psit->rs.as<R>(), pl, out, c->halo.as<R>(), hcs, (R)sp->qbm, (R)sp->dt,
                       (R)dex, c->skip, psi ? psi->rs.as<R>() : nullptr, (R)sp->q_value);
    }
    QP_LAUNCH_CHECK();
    return QP_OK;
}

// the default shape, by the bands of a tile
template <typename R, bool ADD>
static int amjdp_banded(qp_species *sp, const qp_field2d *ef, const qp_field2d *bf,
                        const qp_field2d *psit, double dex, const DepOut<R> &out,
                        const qp_field2d *psi, int bands)
{
    return bands == 4   ? amjdp_v<R, 0, 4, ADD>(sp, ef, bf, psit, dex, out, psi)
           : bands == 2 ? amjdp_v<R, 0, 2, ADD>(sp, ef, bf, psit, dex, out, psi)
                        : amjdp_v<R, 0, 1, ADD>(sp, ef, bf, psit, dex, out, psi);
}

template <typename R>
static int amjdp_out(qp_species *sp, const qp_field2d *ef, const qp_field2d *bf,
                     const qp_field2d *psit, double dex, const DepOut<R> &out,
                     const qp_field2d *psi = nullptr, BorderJob *job = nullptr)
{
    int rc, bands = 1;
    switch (sp->ctx->tune[QP_TUNE_AMJDP]) {
    case 1: rc = amjdp_v<R, 1>(sp, ef, bf, psit, dex, out, psi); break;
    case 2: rc = amjdp_v<R, 2>(sp, ef, bf, psit, dex, out, psi); break;
    case 3: rc = amjdp_v<R, 3>(sp, ef, bf, psit, dex, out, psi); break;
    case 4: rc = amjdp_v<R, 4>(sp, ef, bf, psit, dex, out, psi); break;
    case 5: rc = amjdp_v<R, 5>(sp, ef, bf, psit, dex, out, psi); break;
    case 6: rc = amjdp_v<R, 6>(sp, ef, bf, psit, dex, out, psi); break;
    case 7: rc = amjdp_v<R, 7>(sp, ef, bf, psit, dex, out, psi); break;
    case 8: rc = amjdp_v<R, 8>(sp, ef, bf, psit, dex, out, psi); break;
    case 9: rc = amjdp_v<R, 9>(sp, ef, bf, psit, dex, out, psi); break;
    case 10: rc = amjdp_v<R, 10>(sp, ef, bf, psit, dex, out, psi); break;
    case 11: rc = amjdp_v<R, 11>(sp, ef, bf, psit, dex, out, psi); break;
    case 12: rc = amjdp_v<R, 12>(sp, ef, bf, psit, dex, out, psi); break;
    case 13: rc = amjdp_v<R, 13>(sp, ef, bf, psit, dex, out, psi); break;
    case 14: rc = amjdp_v<R, 14>(sp, ef, bf, psit, dex, out, psi); break;
    default:
        bands = deposit_bands(sp->ctx);
        rc = out.inner[0] ? amjdp_banded<R, true>(sp, ef, bf, psit, dex, out, psi, bands)
                          : amjdp_banded<R, false>(sp, ef, bf, psit, dex, out, psi, bands);
        break;
    }
    if (rc) return rc;
    return deposit_border<R>(sp->ctx, out, 8, 1, nullptr, bands, job);
}

// qdp_species2d with the slice's additions fused into the deposit
// (species2d_class.f03:166-185): this%q = deposit; q = this%q + q;
// q = qn + q.  first: q holds nothing yet (the slice loop zeroed it).  bp: the
// beam plane to convert beside it (or null); halo: the tile-border buffer
// (null: the context's).
template <typename R>
static int qdp_fused_t(qp_species *sp, qp_field2d *q, bool first, const BeamPlane *bp,
                       BorderJob *job, void *halo)
{
    R *qp = q->rs.as<R>();
    DepOut<R> o{};
    o.p[0] = qp;
    o.inner[0] = first ? nullptr : qp;
    o.outer[0] = sp->qn->rs.as<R>();
    o.p2[0] = sp->q->rs.as<R>();
    o.scale = o.scale2 = R(1);
    int rc = deposit_q_out<R>(sp, o, static_cast<R *>(halo), bp, job);
    if (rc) return rc;
    sp->q->state = 0;
    sp->q->gcells = 1;
    q->state = 0;
    return QP_OK;
}

// amjdp_species2d plus the slice loop's scaling (species2d_class.f03:187-218,
// simulation_class.f03:682-685): cu = this%cu + cu (likewise dcu, amu),
// this%cu *= dex, and after the last species cu, amu, dcu *= dex.  Of the
// species' own planes only this%cu(3) is kept (its one later reader, cbq).
template <typename R>
static int amjdp_fused_t(qp_species *sp, const qp_field2d *ef, const qp_field2d *bf,
                         const qp_field2d *psit, qp_field2d *cu, qp_field2d *dcu,
                         qp_field2d *amu, double dex, bool first, bool last,
                         const qp_field2d *psi, BorderJob *job)
{
    const size_t pl = sp->ctx->rplane;
    R *c = cu->rs.as<R>(), *d = dcu->rs.as<R>(), *a = amu->rs.as<R>();
    R *planes[8] = {c, c + pl, c + 2 * pl, d, d + pl, a, a + pl, a + 2 * pl};
    DepOut<R> o{};
    for (int k = 0; k < 8; ++k) {
        o.p[k] = planes[k];
        o.inner[k] = first ? nullptr : planes[k];
    }
    o.p2[2] = sp->cu->rs.as<R>() + 2 * pl;
    o.scale = last ? (R)dex : R(1);
    o.scale2 = (R)dex;
    int rc = amjdp_out<R>(sp, ef, bf, psit, dex, o, psi, job);
    sp->cu->state = 0;
    cu->state = dcu->state = amu->state = 0;
    return rc;
}

// amjdp_species2d's deposit (species2d_class.f03:187-218) into the species' own
// cu, dcu, amu (overwritten)
template <typename R>
static int amjdp_t(qp_species *sp, const qp_field2d *ef, const qp_field2d *bf,
                   const qp_field2d *psit, double dex)
{
    const size_t pl = sp->ctx->rplane;
    R *cu = sp->cu->rs.as<R>(), *dcu = sp->dcu->rs.as<R>(), *amu = sp->amu->rs.as<R>();
    R *planes[8] = {cu, cu + pl, cu + 2 * pl, dcu, dcu + pl, amu, amu + pl, amu + 2 * pl};
    int rc = amjdp_out<R>(sp, ef, bf, psit, dex, dep_plain<R>(planes, 8));
    sp->cu->state = sp->dcu->state = sp->amu->state = 0;
    return rc;
}

// amjdp_species2d's deposit and additions in one: this%cu = deposit * dex, and
// cu = deposit + cu, dcu and amu likewise (species2d_class.f03:187-218)
template <typename R>
static int amjdp_add_t(qp_species *sp, const qp_field2d *ef, const qp_field2d *bf,
                       const qp_field2d *psit, qp_field2d *cu, qp_field2d *dcu, qp_field2d *amu,
                       double dex)
{
    const size_t pl = sp->ctx->rplane;
    R *c = cu->rs.as<R>(), *d = dcu->rs.as<R>(), *a = amu->rs.as<R>();
    R *planes[8] = {c, c + pl, c + 2 * pl, d, d + pl, a, a + pl, a + 2 * pl};
    DepOut<R> o = dep_plain<R>(planes, 8);
    for (int k = 0; k < 8; ++k) o.inner[k] = planes[k];
    for (int k = 0; k < 3; ++k) o.p2[k] = sp->cu->rs.as<R>() + k * pl;
    o.scale2 = (R)dex;
    int rc = amjdp_out<R>(sp, ef, bf, psit, dex, o);
    if (rc) return rc;
    sp->cu->state = 0;
    for (qp_field2d *f : {cu, dcu, amu}) f->gcells = sp->cu->gcells;
    return QP_OK;
}

template <typename R>
static int push_t(qp_species *sp, const qp_field2d *ef, const qp_field2d *bf,
                  const qp_field2d *psit, double dex, bool check, bool raw = false)
{
    qp_ctx *c = sp->ctx;
    const TileGeom g = geom(c);
    const bool scatter = c->tune[QP_TUNE_PUSH] == 1;
    // Blocks of 1024 where every tile has a unit of its own and more particles than
    // a block of 256 takes at once: four waves a SIMD cover each other's waits.
    // FP64, 4 a cell, first and second pass: 64 x 32 10.3 + 11.0 -> 7.3 + 8.3 us,
    // 128^2 10.8 + 12.6 -> 8.2 + 10.3; but 512 tiles (9 a cell) 20 + 36 -> 24 + 38,
    // and 512^2 FP32 (1024 tiles, 4 a cell) 14.6 + 19.3 -> 17.0 + 27.7.
    const bool wide = !scatter && c->ntiles <= c->cus && sp->np > (int64_t)256 * c->ntiles;
    const double fields = 6.0 * (c->nx + 1.0) * (c->ny + 1.0) * sizeof(R);
    const Soa<R> a = soa<R>(sp->a), b = soa<R>(sp->b);
    int *off = sp->off.as<int>(), *off_new = sp->off_new.as<int>();
    {
    // in place: 7 arrays read, 5 written; counting: 7 read
    ProfScope _ps(c, QP_PROF_PUSH, (scatter ? 12.0 : 7.0) * sp->np * sizeof(R) + fields);
    auto kern = scatter ? k_push<R, 0> : wide ? k_push<R, 1, PUSH_WIDE> : k_push<R, 1>;
    hipLaunchKernelGGL(kern, dim3(c->ntiles), dim3(wide ? PUSH_WIDE : 256), 0, c->stream, g, a, b, off, off_new,
                       ef->rs.as<R>(), bf->rs.as<R>(), psit->rs.as<R>(), c->rplane,
                       (R)sp->qbm, (R)sp->dt, (R)dex, sp->key.as<int>(), sp->slot.as<int>(),
                       sp->bins.as<int>(), sp->err.as<int>(), sp->np, 0, raw ? 1 : 0,
                       sp->tot.as<int>());
    }
    QP_LAUNCH_CHECK();
    if (scatter) {
        {
        ProfScope _ps(c, QP_PROF_SORT, 8.0 * (double)c->ntiles * NBINS);
        hipLaunchKernelGGL(k_bin_starts, dim3(c->ncells / 256 + 1), dim3(256), 0, c->stream, g,
                           sp->bins.as<int>(), sp->count.as<int>());
        }
        QP_LAUNCH_CHECK();
        int rc = scan_counts(sp);
        if (rc) return rc;
        {
        ProfScope _ps(c, QP_PROF_SORT, 18.0 * sizeof(R) * (double)sp->np);
        hipLaunchKernelGGL(k_scatter<R>, pgrid(sp->np), dim3(256), 0, c->stream, sp->np, a, b,
                           sp->key.as<int>(), sp->slot.as<int>(), sp->bins.as<int>(), off,
                           c->mx1, c->my1);
        }
        QP_LAUNCH_CHECK();
    } else {
        int *tot = sp->tot.as<int>(), *grp = c->ntiles > 8192 ? tot + c->ntiles : nullptr;
        if (grp) {
            hipLaunchKernelGGL(k_group_totals, dim3((c->ntiles + GROUP - 1) / GROUP), dim3(GROUP),
                               0, c->stream, c->ntiles, tot, grp);
            QP_LAUNCH_CHECK();
        }
        {
        ProfScope _ps(c, QP_PROF_SORT, 8.0 * (double)c->ntiles * NBINS);
        hipLaunchKernelGGL(k_bin_offsets, dim3(c->ntiles), dim3(TCELLS), 0, c->stream, g,
                           sp->bins.as<int>(), tot, grp, off_new);
        }
        QP_LAUNCH_CHECK();
        {
        // 8 arrays read, 8 written at their sorted places
        ProfScope _ps(c, QP_PROF_SORT, (sp->q_uniform ? 14.0 : 16.0) * sp->np * sizeof(R) + fields);
        auto kern = wide ? k_push<R, 2, PUSH_WIDE> : k_push<R, 2>;
        hipLaunchKernelGGL(kern, dim3(c->ntiles), dim3(wide ? PUSH_WIDE : 256), 0, c->stream, g, a, b,
                           off, off_new, ef->rs.as<R>(), bf->rs.as<R>(), psit->rs.as<R>(),
                           c->rplane, (R)sp->qbm, (R)sp->dt, (R)dex, nullptr, nullptr,
                           sp->bins.as<int>(), sp->err.as<int>(), sp->np, sp->q_uniform ? 1 : 0,
                           raw ? 1 : 0, sp->tot.as<int>());
        }
        QP_LAUNCH_CHECK();
        std::swap(sp->off, sp->off_new);
    }
    for (int k = 0; k < 8; ++k) std::swap(sp->a[k], sp->b[k]);
    return check ? check_err(sp, "pmove") : QP_OK;
}

int species_qdp_into(qp_species *sp, qp_field2d *q)
{
    return qp_species_qdp(sp, q);
}

}  // namespace qp

using namespace qp;

#define SPCHECK(sp) QP_REQUIRE((sp) && (sp)->ctx, QP_ERR_ARG, "%s: null species", __func__)
#define DISPATCH(c, fn, ...) ((c)->prec == QP_FP64 ? fn<double>(__VA_ARGS__) : fn<float>(__VA_ARGS__))

extern "C" {

int qp_species_create(qp_ctx *c, const qp_species_params *p, double dt, double s,
                      qp_species **out)
{
    QP_REQUIRE(c && p && out, QP_ERR_ARG, "qp_species_create: null argument");
    QP_REQUIRE(p->ppc[0] >= 1 && p->ppc[1] >= 1 && p->q != 0.0 && p->m != 0.0, QP_ERR_ARG,
               "qp_species_create: bad species parameters");
    qp_species *sp = new qp_species();
    sp->ctx = c;
    sp->p = *p;
    sp->qbm = p->q / p->m;
    sp->dt = dt;
    const int64_t np = (int64_t)(c->nx - 2) * (c->ny - 1) * p->ppc[0] * p->ppc[1];
    int rc = den_factor_at(sp, s);
    if (!rc) rc = DISPATCH(c, alloc_particles, sp, np);
    if (!rc) rc = qp_field2d_create(c, 1, 0, &sp->q);
    if (!rc) rc = qp_field2d_create(c, 1, 0, &sp->qn);
    if (!rc) rc = qp_field2d_create(c, 3, 0, &sp->cu);
    if (!rc) rc = qp_field2d_create(c, 2, 0, &sp->dcu);
    if (!rc) rc = qp_field2d_create(c, 3, 0, &sp->amu);
    if (!rc) rc = DISPATCH(c, renew_t, sp);
    if (rc) { qp_species_destroy(sp); return rc; }
    *out = sp;
    return QP_OK;
}

int qp_species_destroy(qp_species *sp)
{
    if (!sp) return QP_OK;
    if (sp->ctx) (void)hipStreamSynchronize(sp->ctx->stream);
    for (int k = 0; k < 8; ++k) { sp->a[k].release(); sp->b[k].release(); }
    sp->key.release(); sp->slot.release(); sp->count.release(); sp->off.release();
    sp->off_new.release();
    sp->bins.release();
    sp->tot.release();
    sp->scan_tmp.release(); sp->err.release(); sp->radial.release();
    if (sp->h_err) (void)hipHostFree(sp->h_err);
    if (sp->err_ev) (void)hipEventDestroy(sp->err_ev);
    qp_field2d_destroy(sp->q); qp_field2d_destroy(sp->qn); qp_field2d_destroy(sp->cu);
    qp_field2d_destroy(sp->dcu); qp_field2d_destroy(sp->amu);
    delete sp;
    return QP_OK;
}

int qp_species_renew(qp_species *sp, double s)
{
    SPCHECK(sp);
    int rc = den_factor_at(sp, s);
    if (rc) return rc;
    return DISPATCH(sp->ctx, renew_t, sp);
}

int qp_species_set_longitudinal(qp_species *sp, int n, const double *s, const double *fs,
                                double s_now)
{
    SPCHECK(sp);
    QP_REQUIRE(n == 0 || (n >= 2 && s && fs), QP_ERR_ARG,
               "qp_species_set_longitudinal: %d points (0, or at least 2)", n);
    sp->lp_s.assign(s, s + n);
    sp->lp_fs.assign(fs, fs + n);
    return qp_species_renew(sp, s_now);
}

// init_fdist2d_010 / _011 / _012 (fdist2d_class.f03:318-388, 525-590,
// 713-776): lengths to grid units, the centre relative to the box's lower
// corner; then a reload at s_now
int qp_species_set_profile(qp_species *sp, const qp_species_profile *p, double s_now)
{
    SPCHECK(sp);
    QP_REQUIRE(p, QP_ERR_ARG, "qp_species_set_profile: null profile");
    QP_REQUIRE(p->profile == 0 || p->profile == 10 || p->profile == 11 || p->profile == 12,
               QP_ERR_UNSUPPORTED, "qp_species_set_profile: plasma profile %d (0, 10, 11, 12)",
               p->profile);
    const qp_ctx *c = sp->ctx;
    const double dx = c->dex, dy = c->dey;
    if (p->profile == 10)
        QP_REQUIRE(p->inner_radius[0] > 0 && p->inner_radius[1] > 0 && p->outer_radius[0] > 0 &&
                       p->outer_radius[1] > 0,
                   QP_ERR_ARG, "profile 10: radii must be positive");
    if (p->profile == 11)
        QP_REQUIRE(p->width > 0, QP_ERR_ARG, "profile 11: width must be positive");
    if (p->profile == 12) {
        QP_REQUIRE(p->nr >= 2 && p->r && p->fr, QP_ERR_ARG,
                   "profile 12: at least 2 radial points");
    }
    sp->profile = p->profile;
    sp->pcx = (p->center[0] - c->box[0]) / dx;
    sp->pcy = (p->center[1] - c->box[2]) / dy;
    sp->irx = p->inner_radius[0] / dx;
    sp->iry = p->inner_radius[1] / dy;
    sp->orx = p->outer_radius[0] / dx;
    sp->ory = p->outer_radius[1] / dy;
    sp->r0 = p->radius / dx;
    sp->sigr = p->width / dx;
    sp->pr.clear();
    sp->pfr.clear();
    if (p->profile == 12)
        for (int k = 0; k < p->nr; ++k) {
            sp->pr.push_back(p->r[k] / dx);
            sp->pfr.push_back(p->fr[k]);
        }
    if (!sp->pr.empty()) {
        std::vector<double> h(sp->pr);
        h.insert(h.end(), sp->pfr.begin(), sp->pfr.end());
        QP_HIP(hipStreamSynchronize(c->stream));   // no load is reading the old points
        int rc = sp->radial.alloc(h.size() * sizeof(double));
        if (rc) return rc;
        QP_HIP(hipMemcpy(sp->radial.p, h.data(), h.size() * sizeof(double),
                         hipMemcpyHostToDevice));
    }
    return qp_species_renew(sp, s_now);
}

// qdp_species2d (species2d_class.f03:166-185): this%q = folded deposit;
// q = this%q + q; q = qn + q
int qp_species_qdp(qp_species *sp, qp_field2d *q)
{
    SPCHECK(sp);
    QP_REQUIRE(q && q->dim == 1 && q->state == 0, QP_ERR_STATE, "qdp: q must be real space, dim 1");
    int rc = DISPATCH(sp->ctx, qdp_fused_t, sp, q, false, nullptr, nullptr, nullptr);
    if (!rc) q->gcells = sp->qn->gcells;
    return rc;
}

// qp_species_qdp with the deposit's tile-border halo in the library's static
// scratch array instead of the context's buffer: no allocation of any kind.
// Every call on a GPU shares that GPU's array, so calls on one GPU that
// overlap (other threads, or other streams without ordering) race.  The
// halo is fully rewritten by every deposit before it is read, so nothing
// has to be cleared between calls.
int qp_species_qdp_noalloc(qp_species *sp, qp_field2d *q)
{
    SPCHECK(sp);
    QP_REQUIRE(q && q->dim == 1 && q->state == 0, QP_ERR_STATE,
               "qdp_noalloc: q must be real space, dim 1");
    qp_ctx *c = sp->ctx;
    const size_t need = (size_t)c->ntiles * HALO * c->esize;
    QP_REQUIRE(need <= qp::NOALLOC_BYTES, QP_ERR_UNSUPPORTED,
               "qdp_noalloc: %d tiles need %zu B of scratch; the maximum is %zu B "
               "(%zu tiles in this precision)",
               c->ntiles, need, qp::NOALLOC_BYTES, qp::NOALLOC_BYTES / (HALO * c->esize));
    void *halo = qp::noalloc_scratch(c->device);
    QP_REQUIRE(halo, QP_ERR_UNSUPPORTED, "qdp_noalloc: no scratch address for device %d",
               c->device);
    int rc = DISPATCH(c, qdp_fused_t, sp, q, false, nullptr, nullptr, halo);
    if (!rc) q->gcells = sp->qn->gcells;
    return rc;
}

int qp_species_extpsi(qp_species *sp, const qp_field2d *psi, double dex)
{
    SPCHECK(sp);
    QP_REQUIRE(psi && psi->state == 0, QP_ERR_STATE, "extpsi: psi must be real space");
    return DISPATCH(sp->ctx, extpsi_t, sp, psi, dex);
}

// amjdp_species2d (species2d_class.f03:187-218)
int qp_species_amjdp(qp_species *sp, const qp_field2d *ef, const qp_field2d *bf,
                     const qp_field2d *psit, qp_field2d *cu, qp_field2d *amu, qp_field2d *dcu,
                     double dex)
{
    SPCHECK(sp);
    QP_REQUIRE(ef && bf && psit && cu && amu && dcu, QP_ERR_ARG, "amjdp: null field");
    QP_REQUIRE(ef->state == 0 && bf->state == 0 && psit->state == 0, QP_ERR_STATE,
               "amjdp: fields must be real space");
    QP_REQUIRE(ef->dim >= 2 && bf->dim == 3 && cu->dim == 3 && dcu->dim >= 2 && amu->dim == 3,
               QP_ERR_ARG, "amjdp: component counts");
    QP_REQUIRE(cu->state == 0 && dcu->state == 0 && amu->state == 0, QP_ERR_STATE,
               "field op: states are different");
    QP_REQUIRE(dcu->dim == 2, QP_ERR_ARG, "field op: dim mismatch");
    // The additions go with the deposit's stores (four launches less).  Fields that
    // are also inputs of the deposit, or given twice, are added to behind it.
    const qp_field2d *out[3] = {cu, dcu, amu};
    bool apart = cu != dcu && cu != amu && dcu != amu;
    for (const qp_field2d *f : out) apart = apart && f != ef && f != bf && f != psit;
    if (apart) return DISPATCH(sp->ctx, amjdp_add_t, sp, ef, bf, psit, cu, dcu, amu, dex);
    int rc = DISPATCH(sp->ctx, amjdp_t, sp, ef, bf, psit, dex);
    if (!rc) rc = qp_field2d_add(cu, sp->cu, cu, 0, nullptr, nullptr, nullptr);
    if (!rc) rc = qp_field2d_add(dcu, sp->dcu, dcu, 0, nullptr, nullptr, nullptr);
    if (!rc) rc = qp_field2d_add(amu, sp->amu, amu, 0, nullptr, nullptr, nullptr);
    double d = dex;
    if (!rc) rc = qp_field2d_mult(sp->cu, sp->cu, 0, nullptr, nullptr, &d);
    return rc;
}

int qp_species_push(qp_species *sp, const qp_field2d *ef, const qp_field2d *bf,
                    const qp_field2d *psit, double dex)
{
    SPCHECK(sp);
    QP_REQUIRE(ef && bf && psit && ef->state == 0 && bf->state == 0 && psit->state == 0,
               QP_ERR_STATE, "push: fields must be real space");
    return DISPATCH(sp->ctx, push_t, sp, ef, bf, psit, dex, true);
}

// cbq_species2d (species2d_class.f03:399-418)
int qp_species_cbq(qp_species *sp, qp_field3d *q3, int pos)
{
    SPCHECK(sp);
    const int d1[1] = {1}, d3[1] = {3};
    int rc = qp_field2d_add(sp->q, sp->q, sp->cu, 1, d1, d1, d3);
    if (!rc) rc = qp_field2d_fftrk(sp->q, 1);
    if (!rc) rc = qp_field2d_smooth(sp->q, sp->q);
    if (!rc) rc = qp_field2d_fftkr(sp->q, 1);
    if (!rc && q3) rc = qp_field2d_cb(sp->q, q3, pos, 1, d1, d1);
    return rc;
}

}  // extern "C"

namespace qp {
// the first plane of the species' 3-D charge at a (re)load on the first
// stage (species2d_class.f03:107-113, 151-157): q = the fresh plasma's
// folded deposit (-qn), smoothed, into plane 1
int species_q3_initial(qp_species *sp, qp_field3d *q3)
{
    SPCHECK(sp);
    const int d1[1] = {1};
    double m1 = -1.0;
    int rc = qp_field2d_mult(sp->q, sp->qn, 0, nullptr, nullptr, &m1);
    if (!rc) rc = qp_field2d_fftrk(sp->q, 1);
    if (!rc) rc = qp_field2d_smooth(sp->q, sp->q);
    if (!rc) rc = qp_field2d_fftkr(sp->q, 1);
    if (!rc && q3) rc = qp_field2d_cb(sp->q, q3, 1, 1, d1, d1);
    return rc;
}
}  // namespace qp
extern "C" {

int qp_species_count(const qp_species *sp, int64_t *np)
{
    SPCHECK(sp);
    *np = sp->np;
    return QP_OK;
}

}  // extern "C"

static int host_cell_counts(const qp_species *sp, std::vector<int> &off);

template <typename R>
static int download_t(const qp_species *sp, double *part, int64_t ld)
{
    qp_ctx *c = sp->ctx;
    std::vector<R> h((size_t)sp->np);
    // FP32 positions are relative to their tile's origin: the tile of each
    // particle comes from the cell offsets (the records are sorted by tile)
    std::vector<double> ox, oy;
    if (TileRel<R>::on) {
        std::vector<int> off;
        int rc = host_cell_counts(sp, off);
        if (rc) return rc;
        ox.resize((size_t)sp->np);
        oy.resize((size_t)sp->np);
        for (int t = 0; t < c->ntiles; ++t)
            for (int i = off[(size_t)t * TCELLS]; i < off[(size_t)(t + 1) * TCELLS]; ++i) {
                ox[i] = (double)((t % c->mx1) * TILE);
                oy[i] = (double)((t / c->mx1) * TILE);
            }
    }
    for (int k = 0; k < 8; ++k) {
        QP_HIP(hipMemcpyAsync(h.data(), sp->a[k].p, h.size() * sizeof(R), hipMemcpyDeviceToHost,
                              c->stream));
        QP_HIP(hipStreamSynchronize(c->stream));
        // words 6 and 7 of an FP32 record are held as deviations from 1
        const double base = (P67Dev<R>::on && (k == 5 || k == 6)) ? 1.0 : 0.0;
        if (TileRel<R>::on && k < 2) {
            const std::vector<double> &o = k == 0 ? ox : oy;
            for (int64_t i = 0; i < sp->np; ++i) part[k + 8 * i] = (double)h[i] + o[i];
        } else {
            for (int64_t i = 0; i < sp->np; ++i) part[k + 8 * i] = (double)h[i] + base;
        }
    }
    (void)ld;
    return QP_OK;
}

extern "C" {

int qp_species_download(const qp_species *sp, double *part, int64_t ld)
{
    SPCHECK(sp);
    QP_REQUIRE(part && ld >= sp->np, QP_ERR_ARG, "qp_species_download: bad buffer");
    return sp->ctx->prec == QP_FP64 ? download_t<double>(sp, part, ld)
                                    : download_t<float>(sp, part, ld);
}

}  // extern "C"

template <typename R>
static int upload_t(qp_species *sp, const double *part, int64_t np)
{
    qp_ctx *c = sp->ctx;
    std::vector<R> h((size_t)np);
    // FP32: cell keys from the positions in grid units, and the positions
    // relative to their tile (in FP64, then rounded)
    std::vector<int> hkeys;
    if (TileRel<R>::on) {
        hkeys.resize((size_t)np);
        for (int64_t i = 0; i < np; ++i) {
            const double x = part[8 * i], y = part[1 + 8 * i];
            QP_REQUIRE(x >= 0.0 && x < (double)c->nx && y >= 0.0 && y < (double)c->ny,
                       QP_ERR_CHECK, "particle load: particle position outside the grid");
            hkeys[i] = host_cell_key((int)x, (int)y, c->mx1);
        }
    }
    for (int k = 0; k < 8; ++k) {
        const double base = (P67Dev<R>::on && (k == 5 || k == 6)) ? 1.0 : 0.0;
        if (TileRel<R>::on && k < 2)
            for (int64_t i = 0; i < np; ++i) {
                const double v = part[k + 8 * i];
                h[i] = (R)(v - (double)((int)v & ~(TILE - 1)));
            }
        else
            for (int64_t i = 0; i < np; ++i) h[i] = (R)(part[k + 8 * i] - base);
        QP_HIP(hipMemcpyAsync(sp->a[k].p, h.data(), h.size() * sizeof(R), hipMemcpyHostToDevice,
                              c->stream));
        QP_HIP(hipStreamSynchronize(c->stream));
    }
    sp->np = np;
    // a uniform charge (compared as stored) lets the kernels skip q
    bool uniform = true;
    const R q0 = np ? (R)part[7] : R(0);
    for (int64_t i = 1; uniform && i < np; ++i) uniform = (R)part[7 + 8 * i] == q0;
    int rc = rebin_unsorted<R>(sp, TileRel<R>::on ? &hkeys : nullptr);
    if (rc) return rc;
    return set_q_uniform(sp, uniform, (double)q0);
}

extern "C" {

int qp_species_upload(qp_species *sp, const double *part, int64_t np, int64_t ld)
{
    SPCHECK(sp);
    QP_REQUIRE(part && np >= 0 && ld >= np, QP_ERR_ARG, "qp_species_upload: bad buffer");
    QP_REQUIRE((size_t)np * sp->ctx->esize <= sp->a[0].bytes, QP_ERR_ARG,
               "qp_species_upload: %lld particles exceed the capacity", (long long)np);
    return sp->ctx->prec == QP_FP64 ? upload_t<double>(sp, part, np)
                                    : upload_t<float>(sp, part, np);
}

static int host_cell_counts(const qp_species *sp, std::vector<int> &off)
{
    qp_ctx *c = sp->ctx;
    off.resize((size_t)c->ncells + 1);
    QP_HIP(hipMemcpyAsync(off.data(), sp->off.p, off.size() * 4, hipMemcpyDeviceToHost, c->stream));
    QP_HIP(hipStreamSynchronize(c->stream));
    return QP_OK;
}

int qp_species_cell_counts(const qp_species *sp, int32_t *counts)
{
    SPCHECK(sp);
    std::vector<int> off;
    int rc = host_cell_counts(sp, off);
    if (rc) return rc;
    qp_ctx *c = sp->ctx;
    for (int cy = 0; cy < c->ny; ++cy)
        for (int cx = 0; cx < c->nx; ++cx) {
            int k = ((cy / TILE) * c->mx1 + cx / TILE) * TCELLS + (cy % TILE) * TILE + cx % TILE;
            counts[(size_t)cy * c->nx + cx] = off[k + 1] - off[k];
        }
    return QP_OK;
}

int qp_species_tile_counts(const qp_species *sp, int32_t *kpic)
{
    SPCHECK(sp);
    std::vector<int> off;
    int rc = host_cell_counts(sp, off);
    if (rc) return rc;
    for (int t = 0; t < sp->ctx->ntiles; ++t) kpic[t] = off[(t + 1) * TCELLS] - off[t * TCELLS];
    return QP_OK;
}

}  // extern "C"

// entry points used by the slice driver without the per-call error sync
namespace qp {
// ef holds grad(psi) still (see k_push)
int species_push_nocheck(qp_species *sp, const qp_field2d *ef, const qp_field2d *bf,
                         const qp_field2d *psit, double dex)
{
    return DISPATCH(sp->ctx, push_t, sp, ef, bf, psit, dex, false, true);
}
int species_check(qp_species *sp) { return check_err(sp, "pmove"); }

// The push leaves the particles in the alternate arrays and swaps the
// host's buffer pointers (and, when it re-sorts in place, the cell offsets).
// A captured slice repeats the device side only; these let its caller keep
// the host side in step: which buffer holds the particles, and one swap.
const void *species_buffer_key(const qp_species *sp) { return sp->a[0].p; }
void species_flip(qp_species *sp, bool offsets)
{
    if (offsets) std::swap(sp->off, sp->off_new);
    for (int k = 0; k < 8; ++k) std::swap(sp->a[k], sp->b[k]);
}

// The slice loop does not wait for the move check of each push: the error
// word is copied to pinned memory behind the push, and a later slice (or the
// end of the step, which waits) reports it.  The words to copy are given to
// the kernel that ends the slice (species_err_words, then species_check_mark
// behind it); species_check_post copies them by a launch of its own.
void species_err_words(qp_species *sp, const int **err, int **h_err)
{
    *err = sp->err.as<int>();
    *h_err = sp->h_err;
}
int species_check_mark(qp_species *sp)
{
    QP_HIP(hipEventRecord(sp->err_ev, sp->ctx->stream));
    sp->err_pending = true;
    return QP_OK;
}
int species_check_post(qp_species *sp, int slice)
{
    qp_ctx *c = sp->ctx;
    hipLaunchKernelGGL(k_post_err, dim3(1), dim3(64), 0, c->stream, sp->err.as<int>(), sp->h_err,
                       slice);
    QP_LAUNCH_CHECK();
    return species_check_mark(sp);
}

// The move check of the slices posted so far, once their push has run
// (wait: block until it has).  The error names the slice whose push moved a
// particle too far; the slices after it were computed from misplaced
// particles and are invalid, like everything after the reference's stop.
int species_check_poll(qp_species *sp, bool wait)
{
    if (!sp->err_pending) return QP_OK;
    if (wait) QP_HIP(hipEventSynchronize(sp->err_ev));
    else if (hipEventQuery(sp->err_ev) != hipSuccess) return QP_OK;
    sp->err_pending = false;
    const int h = sp->h_err[0], slice = sp->h_err[1];
    if (!h) return QP_OK;
    sp->h_err[0] = sp->h_err[1] = 0;
    QP_HIP(hipMemsetAsync(sp->err.p, 0, sizeof(int), sp->ctx->stream));
    if (h >= (1 << 30))
        set_error("pmove: particle position outside the grid (push of slice %d)", slice);
    else if (h >= (1 << 29))
        set_error("pmove: the push's two passes disagree (push of slice %d)", slice);
    else
        set_error("pmove: particle left its tile by more than one tile (tile %d, push of "
                  "slice %d)", h, slice);
    return QP_ERR_CHECK;
}

int species_qdp_fused(qp_species *sp, qp_field2d *q, bool first, const BeamPlane *bp,
                      BorderJob *job)
{
    return DISPATCH(sp->ctx, qdp_fused_t, sp, q, first, bp, job, nullptr);
}

int species_amjdp_fused(qp_species *sp, const qp_field2d *ef, const qp_field2d *bf,
                        const qp_field2d *psit, qp_field2d *cu, qp_field2d *dcu, qp_field2d *amu,
                        double dex, bool first, bool last, const qp_field2d *psi, BorderJob *job)
{
    return DISPATCH(sp->ctx, amjdp_fused_t, sp, ef, bf, psit, cu, dcu, amu, dex, first, last,
                    psi, job);
}
}  // namespace qp
