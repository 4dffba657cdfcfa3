// The field solve of the slice loop with the y transforms and the k-space
// arithmetic between them in one kernel (k_mid), and the x transforms around
// it reading or writing transposed planes (k_fft_xt): three launches in place
// of two transforms of two or three launches each and the k-space kernel.
//
//   forward x  rows y of the real planes -> scratch planes [kx][y]
//   mid        per pair of kx rows: y transforms of every component, the
//              modes' arithmetic (qp_pass.h), the inverse y transforms
//   inverse x  scratch planes [kx][y] -> rows y of the real planes
//
// The arithmetic is that of the separate transforms and k-space kernels, value
// by value and with the same fused multiply-adds, so the fields are theirs bit
// for bit.  Only rows of one kx meet in a mode, so no planes cross memory
// between the two y transforms.  The field solves of a
// slice (4.2 to 5.25 passes) took, with the separate kernels and with these:
//   512^2 FP32   334 -> 243 us      1024^2 FP32  724 -> 601 us
//   1024^2 FP64  511 -> 451 us (two passes)
//   128^2 FP64   a whole slice of one species, two passes, 29 -> 16 launches
//                (with what they let the other kernels take over)
//
// Which grids: both sides up to 1024 (fused_fields).  A row pair of all eight
// components has to fit the 160 KB of LDS for the exchange between the
// transforms and the modes: 8 (ny + 1) pairs, 66 KB in FP32 and 131 KB in FP64
// at ny = 1024.
#include "qp_border.h"
#include "qp_fft.h"
#include "qp_pass.h"

namespace qp {

template <typename R> struct XtSet {
    const R *src[8];
    R *dst[8];
};

// A barrier that orders LDS alone: loads and stores of memory stay in flight.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// 16 bytes of Reals
template <typename R> struct alignas(16) Quad {
    R v[16 / sizeof(R)];
};

// Shape of k_fft_xt: FB row pairs per workgroup, so that the transposed side
// moves 2 FB Reals (16 to 256 bytes) of a column at a time; workgroups next to
// each other complete its cache lines in one L2.  Small ones: their waits at
// barriers cover each other.  512^2 FP32, forward and inverse: 16 rows (1024
// threads) 11.8 and 8.9 us, 8 rows 10.1 and 7.2; 1024^2 8 rows 27.4 and 17.4,
// 4 rows 26.9 and 17.1; 128^2 FP64 16 rows 8.4 and 5.2, 8 rows 7.6 and 5.0.
template <typename R, int L> struct XtShape {
    static constexpr int PS = pad_shift<R>();
    using S = FftShape<L, PS>;
    static constexpr int FB = S::TF == 4         ? 16   // one whole wave
                              : S::TF * 8 <= 128 ? 8
                              : S::TF * 4 <= 512 ? 4
                                                 : 2;
    static constexpr int BS = FB * S::TF;
    static constexpr int ROWS = 2 * FB;        // rows per workgroup
    static constexpr int SW = ROWS + 2;        // row pitch of the staging area
    static constexpr int V = 16 / sizeof(R);   // Reals per 16-byte access
    static constexpr int CH = ROWS / V;        // accesses per column piece
    static constexpr size_t LDS = (size_t)FB * S::LDSM * sizeof(cplx<R>);
    static_assert((size_t)(S::N + 1) * SW * sizeof(R) <= LDS, "staging fits the FFT's area");
    static_assert(LDS <= 81920, "two workgroups on a CU");
    // the last workgroup's rows go on past ny; its columns stay in the pitch,
    // which is the next multiple of PITCH above ny
    static_assert(PITCH % ROWS == 0, "whole workgroups of rows in the pitch");
};

// Up to this nx the forward x transforms form the border sums of the deposit in
// front of them (a launch less).  The two launches against the one: 128^2 FP64
// 4.4 + 4.9 us, 7.6; 256 x 512 FP32 5.4 + 6.0, 8.9; 512^2 FP32 5.4 + 10.1, 14.0;
// but 1024^2 11.7 + 26.9, 39.6, and in FP64 14.2 + 39.8, 58.3: there the blocks
// of whole border rows wait longer than a kernel of their own does.
constexpr int BORDER_MAX = 512;

// x transforms of the rows of every component of the batch (grid.y).  INV =
// false: rows y of src (pitch ld_src) to columns y of dst ([kx][y], pitch
// ld_dst).  INV = true: columns y of src to rows y of dst, row 0 also to row
// guard_row.  The transposed side goes through LDS in pieces of ROWS Reals per
// kx, so it takes no pass of its own over memory.  zero_row: a row known to be
// zero (the deposits' folded guard row; -1: none), whose workgroup, when it has
// no other row, stores the zeros without a transform.  Workgroups next to each
// other in y share cache lines on the transposed side; block b takes group
// (b mod 8) (gridDim.x / 8) + b / 8, which puts them on one XCD.
template <typename R, int L, bool INV>
__global__ void __launch_bounds__((XtShape<R, L>::BS))
k_fft_xt(XtSet<R> cs, int nrows, int ld_src, int ld_dst, int types, R scale,
         const cplx<R> *__restrict__ W, int guard_row, int zero_row, const int *skip, ResJob rj,
         BorderArgs<R> bd)
{
    using X = XtShape<R, L>;
    using S = typename X::S;
    constexpr int N = S::N, TF = S::TF, BS = X::BS, SW = X::SW, V = X::V, CH = X::CH;
    if (skip && *skip) {
        // see k_fft_rows: the converged flag is passed on
        if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0 && rj.nblk > 0 && rj.flag_out)
            *rj.flag_out = 1;
        return;
    }
    if (blockIdx.x == 0 && blockIdx.y == 0) run_res_job(rj);
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const int comp = blockIdx.y, tid = threadIdx.x;
    const int type = (types >> comp) & 1;
    const int f = tid / TF, t = tid % TF;
    const int y0 = ((blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3)) * X::ROWS;
    if (y0 >= nrows) return;
    const int ra = y0 + 2 * f;
    const bool live = ra < nrows, hb = ra + 1 < nrows;
    cplx<R> *buf = reinterpret_cast<cplx<R> *>(smem_raw) + f * S::LDSM;
    R *stg = reinterpret_cast<R *>(smem_raw);
    const R *src = cs.src[comp];
    R *dst = cs.dst[comp];
    // 16-byte pieces of the transposed planes: the pieces of kx < N are spread
    // evenly over the threads, those of kx = N go to the first CH threads
    constexpr int K = (N * CH + BS - 1) / BS;
    static_assert(N * CH % BS == 0 || N * CH < BS, "whole rounds of pieces");
    constexpr bool BORDER = !INV && N <= BORDER_MAX;
    const bool border = BORDER && comp >= bd.first && comp < bd.first + bd.n;
    const int bc = border ? comp - bd.first : 0;
    if (!INV && y0 == zero_row && nrows == zero_row + 1) {
        for (int it = tid; it <= N; it += BS) {
            dst[(size_t)it * ld_dst + y0] = R(0);
            if (border) dep_store(bd.out, bc, (size_t)y0 * ld_src + it, R(0));
        }
        return;
    }
    cplx<R> v[8], z[4], zn;
    Twiddles<R, L> tw;
    if (!INV) {
        R la[8], lb[8];
        const R *sa = live ? src + (size_t)ra * ld_src : src;
        const R *sb = live && hb ? sa + ld_src : sa;
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const int e = ext_pos<L>(t + r * TF);
            la[r] = at(sa, e);
            lb[r] = at(sb, e);
        }
        tw.load(W, t);
        if (BORDER && border) {
            // the deposit's border nodes in these rows, all nodes of a row that is
            // a multiple of 2^sh and every 16th of the others: formed here, stored
            // to the plane and handed on through LDS
            constexpr int NC = N / TILE + 1;
            const R *halo = bd.halo + bc * bd.halo_cs;
            const int nr = min(X::ROWS, nrows - y0), sh = bd.sh, low = (1 << sh) - 1;
            const int top = -y0 & low;                       // first whole row
            const int nw = top < nr ? ((nr - 1 - top) >> sh) + 1 : 0;
            const int items = nw * (N + 1) + X::ROWS * NC;
            for (int it = tid; it < items; it += BS) {
                int i, x;
                if (it < nw * (N + 1)) {
                    const int w = it / (N + 1);
                    i = top + (w << sh);
                    x = it - w * (N + 1);
                } else {
                    // rows fastest: a tile's side is contiguous in the buffer
                    const int k = it - nw * (N + 1);
                    i = k % X::ROWS;
                    x = k / X::ROWS * TILE;
                    if (i >= nr) continue;
                    if (((y0 + i) & low) == 0) continue;
                }
                const R val = border_node<R>(bd.g, halo, sh, bd.fold, x, y0 + i);
                stg[i * (N + 1) + x] =
                    dep_store(bd.out, bc, (size_t)(y0 + i) * ld_src + x, val);
            }
            lds_barrier();
            const bool wa = (ra & low) == 0, wb = ((ra + 1) & low) == 0;
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                const int e = ext_pos<L>(t + r * TF);
                const bool col = e % TILE == 0;
                if (live && (wa || col)) la[r] = stg[2 * f * (N + 1) + e];
                if (hb && (wb || col)) lb[r] = stg[(2 * f + 1) * (N + 1) + e];
            }
            lds_barrier();   // buf overwrites the staging area
        }
#pragma unroll
        for (int r = 0; r < 8; ++r)
            v[r] = ext_value<R, L>(type, t + r * TF, live ? la[r] : R(0),
                                   live && hb ? lb[r] : R(0));
    } else {
        Quad<R> q[K], qn;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int it = tid + k * BS;
            if (N * CH % BS == 0 || it < N * CH)
                q[k] = *reinterpret_cast<const Quad<R> *>(src + (size_t)(it / CH) * ld_src + y0 +
                                                          (it % CH) * V);
        }
        if (tid < CH) qn = *reinterpret_cast<const Quad<R> *>(src + (size_t)N * ld_src + y0 + tid * V);
        tw.load(W, t);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int it = tid + k * BS;
            if (N * CH % BS == 0 || it < N * CH)
#pragma unroll
                for (int i = 0; i < V; ++i) stg[(it / CH) * SW + (it % CH) * V + i] = q[k].v[i];
        }
        if (tid < CH)
#pragma unroll
            for (int i = 0; i < V; ++i) stg[N * SW + tid * V + i] = qn.v[i];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const cplx<R> p = *reinterpret_cast<const cplx<R> *>(
                stg + ext_pos<L>(t + r * TF) * SW + 2 * f);
            v[r] = ext_value<R, L>(type, t + r * TF, live ? p.x : R(0), live && hb ? p.y : R(0));
        }
        __syncthreads();   // buf overwrites the staging area
    }
    fft_core<R, L, X::PS>(v, buf, t, tw, z, zn);
    const R half = scale * R(0.5);
    if (INV) {
        if (!live) return;
        R *da = dst + (size_t)ra * ld_dst, *db = da + ld_dst;
        R *dg = guard_row >= 0 && ra == 0 ? dst + (size_t)guard_row * ld_dst : nullptr;
        auto emit = [&](int k, cplx<R> x) {
            const cplx<R> o = row_values<R, L>(type, k, x, half);
            at(da, k) = o.x;
            if (hb) at(db, k) = o.y;
            if (dg) at(dg, k) = o.x;
        };
#pragma unroll
        for (int i = 0; i < 4; ++i) emit(t + i * TF, z[i]);
        if (t == 0) emit(N, zn);
        return;
    }
    __syncthreads();   // the staging area overwrites buf
    auto stage = [&](int k, cplx<R> x) {
        *reinterpret_cast<cplx<R> *>(stg + k * SW + 2 * f) = row_values<R, L>(type, k, x, half);
    };
#pragma unroll
    for (int i = 0; i < 4; ++i) stage(t + i * TF, z[i]);
    if (t == 0) stage(N, zn);
    __syncthreads();
    // columns y0 .. y0 + ROWS - 1 lie within the pitch (XtShape)
    auto put = [&](int kx, int c) {
        Quad<R> q;
#pragma unroll
        for (int i = 0; i < V; ++i) q.v[i] = stg[kx * SW + c * V + i];
        *reinterpret_cast<Quad<R> *>(dst + (size_t)kx * ld_dst + y0 + c * V) = q;
    };
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int it = tid + k * BS;
        if (N * CH % BS == 0 || it < N * CH) put(it / CH, it % CH);
    }
    if (tid < CH) put(N, tid);
}

// What k_mid reads and writes.  Planes [kx][ky] (or [kx][y]) with pitch ldk,
// cs elements per component.
template <typename R> struct MidArgs {
    int nx, ldk;
    size_t cs;
    const R *src;              // forward components, cs apart, after the x pass
    R *dst;                    // inverse components, cs apart, before the x pass
    const cplx<R> *W;
    const R *ffg, *ffs;
    R *cu, *dcu, *amu, *epw, *epwb;                   // k planes
    R *qb, *qe, *psi, *fxy, *ehist, *ehist2;         // k planes of the front
    R aa, idex, dex;
    double *partial;           // pass: per-block residual sums
    int *flags;                // front: cleared
    int seed;
    const int *seed_hist, *skip;
};

// The arithmetic of mode (kx, ky): in[] are the forward components' values
// (pass: cu 3, dcu 2, amu 3; front: qb, qe), out[] the inverse components'
// (pass: psit, bxyz 3; front: fxy 2, psi, psit, bxyz 3).  The planes that keep
// k values are written here, except those of in[] itself and, being functions
// of what is kept, psit's and bxyz's (the end of the slice writes them).
template <typename R, int N, bool FRONT, int NF, int NI>
__device__ __forceinline__ void do_mode(const MidArgs<R> &a, int kx, int ky, int seed,
                                        const R (&in)[NF], R (&out)[NI], double &num, double &den)
{
    const size_t cs = a.cs;
    const unsigned m = (unsigned)kx * a.ldk + ky;
    const bool tab = kx < a.nx && ky < N;
    const bool inner = tab && kx > 0 && ky > 0;
    const unsigned ti = tab ? (unsigned)kx * N + ky : 0;
    const R fg = tab ? at(a.ffg, ti) : R(0), fs = tab ? at(a.ffs, ti) : R(0);
    const R dkx = dk<R>(a.nx, kx), dky = dk<R>(N, ky);
    R e1 = at(a.epw, m), e2 = at(a.epw + cs, m);
    R c1, c2, b1, b2;
    if constexpr (FRONT) {
        c1 = at(a.cu, m);
        c2 = at(a.cu + cs, m);
        // elf (MPPOISD22), pot (MPPOTPD2), grad (MPPGRADFD2)
        b1 = b2 = R(0);
        R p = R(0), f1 = R(0), f2 = R(0);
        if (inner) {
            const R at1 = fg * fs;
            const R at3 = -at1 * in[0];
            b1 = dkx * at3;
            b2 = dky * at3;
            p = fg * in[1];
            f1 = dkx * p;
            f2 = dky * p;
        }
        at(a.epwb, m) = b1;
        at(a.epwb + cs, m) = b2;
        at(a.psi, m) = p;
        at(a.fxy, m) = f1;
        at(a.fxy + cs, m) = f2;
        out[0] = f1;
        out[1] = f2;
        out[2] = p;
        if (seed) {
            const R h1 = at(a.ehist, m), h2 = at(a.ehist + cs, m);
            R g1 = R(0), g2 = R(0);
            if (a.ehist2) {
                g1 = at(a.ehist2, m);
                g2 = at(a.ehist2 + cs, m);
                at(a.ehist2, m) = h1;
                at(a.ehist2 + cs, m) = h2;
            }
            at(a.ehist, m) = e1;
            at(a.ehist + cs, m) = e2;
            if (seed >= 2) {
                e1 = seed_mode(seed, e1, h1, g1);
                e2 = seed_mode(seed, e2, h2, g2);
                at(a.epw, m) = e1;
                at(a.epw + cs, m) = e2;
            }
        }
    } else {
        c1 = in[0];
        c2 = in[1];
        b1 = at(a.epwb, m);
        b2 = at(a.epwb + cs, m);
        R d1 = in[3], d2 = in[4], n1, n2;
        corrector_mode(tab, kx, ky, fg, fs, dkx, dky, a.aa, a.idex, in[2], in[5], in[6], in[7], e1,
                       e2, d1, d2, n1, n2);
        at(a.dcu, m) = d1;
        at(a.dcu + cs, m) = d2;
        at(a.epw, m) = n1;
        at(a.epw + cs, m) = n2;
        const double q1 = (double)n1 - (double)e1, q2 = (double)n2 - (double)e2;
        num += q1 * q1 + q2 * q2;
        den += (double)n1 * n1 + (double)n2 * n2;
        e1 = n1;
        e2 = n2;
    }
    constexpr int P = FRONT ? 3 : 0;
    out[P] = psit_mode(inner, fg, dkx, dky, c1, c2, a.dex);
    out[P + 1] = bx_mode(e2, b2, a.dex);
    out[P + 2] = by_mode(e1, b1, a.dex);
    out[P + 3] = bz_mode(tab, kx, ky, fg, fs, dkx, dky, c1, c2) * a.dex;
}

// y types (bit c: cosine) of the forward components, qb, qe sine or cu (S, C,
// S), dcu (S, C), amu (S, S, C), and of the inverse ones, fxy (S, C), psi, psit
// sine, bxyz (C, S, C) or psit, bxyz
template <bool FRONT> struct MidComps {
    static constexpr int NF = FRONT ? 2 : 8, NI = FRONT ? 7 : 4;
    static constexpr int FT = FRONT ? 0 : 0x92, IT = FRONT ? 0x52 : 0xa;
};

// the k plane that keeps forward component c (dcu is written by do_mode)
template <typename R, bool FRONT>
__device__ __forceinline__ R *kept_plane(const MidArgs<R> &a, int c)
{
    if (FRONT) return c == 0 ? a.qb : a.qe;
    return c < 3 ? a.cu + c * a.cs : c < 5 ? nullptr : a.amu + (c - 5) * a.cs;
}

template <typename R> __device__ __forceinline__ int front_seed(const MidArgs<R> &a)
{
    int seed = a.seed;
    if (seed && a.seed_hist) {
        const int n = *a.seed_hist;
        seed = n >= 3 ? 3 : (n >= 2 ? 2 : 1);
    }
    return seed == 3 && !a.ehist2 ? 2 : seed;
}

// the pair of rows (ra, ra + 1) of one component as FFT input; hb: the second
// row exists
template <typename R, int L>
__device__ __forceinline__ void load_pair(const R *sa, int ldk, bool hb, int type, int t,
                                          cplx<R> (&v)[8])
{
    constexpr int TF = FftShape<L>::TF;
    const R *sb = hb ? sa + ldk : sa;
    R la[8], lb[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const int e = ext_pos<L>(t + r * TF);
        la[r] = at(sa, e);
        lb[r] = at(sb, e);
    }
#pragma unroll
    for (int r = 0; r < 8; ++r)
        v[r] = ext_value<R, L>(type, t + r * TF, la[r], hb ? lb[r] : R(0));
}

// Row kx = nx belongs to block 0, beside its own rows: a block of its own would
// be the one that starts a second round on the chip, which nx / 2 blocks fill.
// The tables end at nx - 1, so no mode of it has a value: B_perp becomes zero
// there and, epwb being zero off the modes that elf fills, so do psit and bxyz.
// The forward components that are cosines in x (cu 1, dcu 1, amu 3) are not
// zero and are kept in their k planes (last_row_index, last_row_keep); the
// charges and the other components are sines.
template <typename R, int N, int BS>
__device__ __forceinline__ void last_row_pass(const MidArgs<R> &a, double &num)
{
    const size_t row = (size_t)a.nx * a.ldk, cs = a.cs;
    for (unsigned k = threadIdx.x; k <= N; k += BS) {
        const double e1 = at(a.epw + row, k), e2 = at(a.epw + cs + row, k);
        num += e1 * e1 + e2 * e2;
        at(a.epw + row, k) = at(a.epw + cs + row, k) = R(0);
        at(a.cu + cs + row, k) = at(a.cu + 2 * cs + row, k) = at(a.dcu + cs + row, k) = R(0);
        at(a.amu + row, k) = at(a.amu + cs + row, k) = R(0);
#pragma unroll
        for (int c = 0; c < 4; ++c) at(a.dst + c * cs + row, k) = R(0);
    }
}

__device__ __forceinline__ int last_row_index(int i) { return i == 0 ? 0 : i == 1 ? 3 : 7; }

template <typename R, int L>
__device__ __forceinline__ void last_row_keep(const MidArgs<R> &a, int i, int type, int t,
                                              const cplx<R> (&z)[4], cplx<R> zn)
{
    constexpr int N = FftShape<L>::N, TF = FftShape<L>::TF;
    R *k0 = (i == 0 ? a.cu : i == 1 ? a.dcu : a.amu + 2 * a.cs) + (size_t)a.nx * a.ldk;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        at(k0, t + j * TF) = row_values<R, L>(type, t + j * TF, z[j], R(0.5)).x;
    if (t == 0) k0[N] = row_values<R, L>(type, N, zn, R(0.5)).x;
}

// Row kx = nx of the front: every charge is zero there, and the carried B_perp
// is too after a pass.  One that a caller has put there is carried to bxyz
// (x: cosine in y, y: sine) by direct sums.
template <typename R, int N, int BS>
__device__ void last_row_front(const MidArgs<R> &a, int seed, R *lds)
{
    const size_t row = (size_t)a.nx * a.ldk, cs = a.cs;
    R *e[2] = {lds, lds + N + 1};
    int any = 0;
    __syncthreads();   // lds is free
    for (unsigned k = threadIdx.x; k <= N; k += BS) {
        const R zero[2] = {R(0), R(0)};
        R out[7];
        double x = 0.0, y = 0.0;
        do_mode<R, N, true, 2, 7>(a, a.nx, k, seed, zero, out, x, y);
        at(a.qb + row, k) = at(a.qe + row, k) = R(0);
#pragma unroll
        for (int c = 0; c < 7; ++c) at(a.dst + c * cs + row, k) = R(0);
        e[0][k] = out[4];
        e[1][k] = out[5];
        any |= out[4] != R(0) || out[5] != R(0);
    }
    if (!__syncthreads_or(any)) return;
    for (unsigned y = threadIdx.x; y <= N; y += BS) {
        // 2 C(y) and 2 S(y); W[j] = (cos, -sin)(pi j / N)
        double c = e[0][0] + ((y & 1) ? -e[0][N] : e[0][N]), s = 0.0;
        for (int k = 1; k < N; ++k) {
            const cplx<R> w = a.W[(k * y) & (2 * N - 1)];
            c += 2.0 * (double)e[0][k] * (double)w.x;
            s -= 2.0 * (double)e[1][k] * (double)w.y;
        }
        at(a.dst + 4 * cs + row, y) = (R)c;
        at(a.dst + 5 * cs + row, y) = y == 0 || y == N ? R(0) : (R)s;
    }
}

// per-block sums of the stopping test, in a fixed order
template <int BS>
__device__ __forceinline__ void store_partial(double num, double den, double (*s_sum)[BS / 64 + 1],
                                              double *partial)
{
    const int tid = threadIdx.x;
#pragma unroll
    for (int s = BS < 64 ? BS / 2 : 32; s > 0; s >>= 1) {
        num += __shfl_xor(num, s);
        den += __shfl_xor(den, s);
    }
    if ((tid & 63) == 0) {
        s_sum[0][tid >> 6] = num;
        s_sum[1][tid >> 6] = den;
    }
    __syncthreads();
    if (tid == 0) {
        double x = 0.0, y = 0.0;
        for (int w = 0; w < (BS + 63) / 64; ++w) {
            x += s_sum[0][w];
            y += s_sum[1][w];
        }
        partial[2 * blockIdx.x] = x;
        partial[2 * blockIdx.x + 1] = y;
    }
}

// Component groups of k_mid that transform side by side: all eight of a row
// pair while their LDS leaves room for two workgroups per CU, else four in two
// rounds.
template <typename R, int L> struct MidShape {
    static constexpr int PS = pad_shift<R>();
    using S = FftShape<L, PS>;
    static constexpr int G = S::TF * 8 <= 1024 && 8 * S::LDSM * 2 * sizeof(R) <= 81920 ? 8
                             : S::TF * 4 <= 1024 && S::TF * sizeof(R) <= 1024           ? 4
                                                                                        : 2;
    static constexpr int BS = G * S::TF;
    static constexpr size_t XN = 8 * (size_t)(S::N + 1), BN = (size_t)G * S::LDSM;
    static constexpr size_t LDS = (XN > BN ? XN : BN) * sizeof(cplx<R>);
};

// Between the x passes, for the rows kx = 2 b and 2 b + 1 of block b.
// FRONT = false, a corrector pass (simulation_class.f03:697-709 and the B
// assembly of :677-680): y transforms of cu (3), dcu (2), amu (3); then mode by
// mode bfqp (epw, dcu), psit = pot(div(cu)) (-dex), b = bf(cu), the assembly of
// bxyz and the FP64 sums of the stopping test; then the inverse y transforms
// of psit and bxyz.
// FRONT = true, the start of a slice (:650-680): y transforms of the beam's and
// the plasma's charge; epwb = elf(qb), psi = pot(qe), fxy = grad(psi), the
// corrector seed (as k_pass) and the predictor's psit and bxyz from the carried
// current; then the inverse y transforms of fxy, psi, psit and bxyz.
// For ny < 1024: a group of TF threads transforms one component, and the
// results meet in LDS as pairs (row 2b, row 2b + 1) per component and mode.
template <typename R, int L, bool FRONT>
__global__ void __launch_bounds__((MidShape<R, L>::BS)) k_mid(MidArgs<R> a)
{
    using H = MidShape<R, L>;
    using S = typename H::S;
    using C = MidComps<FRONT>;
    constexpr int N = S::N, TF = S::TF, G = H::G, BS = H::BS, NF = C::NF, NI = C::NI;
    if (a.skip && *a.skip) return;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    __shared__ double s_sum[2][BS / 64 + 1];
    cplx<R> *X = reinterpret_cast<cplx<R> *>(smem_raw);   // [component][N + 1]
    const int tid = threadIdx.x, g = tid / TF, t = tid % TF;
    cplx<R> *buf = X + g * S::LDSM;
    const int ra = 2 * blockIdx.x;
    const size_t row = (size_t)ra * a.ldk, cs = a.cs;
    const bool first = blockIdx.x == 0;
    if (FRONT && first)
        for (int k = tid; k < FLAG_WORDS; k += BS) a.flags[k] = 0;

    // forward y transforms
    constexpr int RF = (NF + G - 1) / G;
    {
    cplx<R> o[RF][4], on[RF];
#pragma unroll
    for (int q = 0; q < RF; ++q) {
        const int c = q * G + g, type = (C::FT >> c) & 1;
        cplx<R> v[8], z[4], zn;
        Twiddles<R, L> tw;
        if (c < NF) {
            load_pair<R, L>(a.src + c * cs + row, a.ldk, true, type, t, v);
        } else {
#pragma unroll
            for (int r = 0; r < 8; ++r) v[r] = {R(0), R(0)};
        }
        tw.load(a.W, t);
        if (q) __syncthreads();
        fft_core<R, L, H::PS>(v, buf, t, tw, z, zn);
#pragma unroll
        for (int i = 0; i < 4; ++i) o[q][i] = row_values<R, L>(type, t + i * TF, z[i], R(0.5));
        on[q] = row_values<R, L>(type, N, zn, R(0.5));
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < RF; ++q) {
        const int c = q * G + g;
        if (c >= NF) break;
        R *k0 = kept_plane<R, FRONT>(a, c);
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            if (i == 4 && t) break;
            const int k = t + i * TF;
            const cplx<R> p = i < 4 ? o[q][i < 4 ? i : 0] : on[q];
            X[c * (N + 1) + k] = p;
            if (k0) {
                at(k0 + row, k) = p.x;
                at(k0 + row + a.ldk, k) = p.y;
            }
        }
    }
    }
    __syncthreads();

    // the modes.  With G = 8 the two rows go to different threads.
    constexpr int RS = G >= 8 ? 2 : 1;
    const int seed = FRONT ? front_seed(a) : 0;
    {
    double num = 0.0, den = 0.0;
    const int r0 = RS == 2 ? tid / N : 0, r1 = RS == 2 ? r0 + 1 : 2;
    constexpr int KS = RS == 2 ? N : BS;
    for (int ky = tid % KS; ky <= N; ky += KS) {
        for (int rr = r0; rr < r1; ++rr) {
            R in[NF], out[NI];
#pragma unroll
            for (int c = 0; c < NF; ++c) {
                const cplx<R> p = X[c * (N + 1) + ky];
                in[c] = rr ? p.y : p.x;
            }
            do_mode<R, N, FRONT, NF, NI>(a, ra + rr, ky, seed, in, out, num, den);
#pragma unroll
            for (int c = 0; c < NI; ++c) {
                cplx<R> *p = X + c * (N + 1) + ky;
                if (rr) p->y = out[c];
                else p->x = out[c];
            }
        }
    }
    if (!FRONT) {
        if (first) last_row_pass<R, N, BS>(a, num);
        store_partial<BS>(num, den, s_sum, a.partial);
    }
    }
    __syncthreads();

    // inverse y transforms: every round's input leaves LDS before buf is used
    constexpr int RI = (NI + G - 1) / G;
    // the last row's three components: by groups without an inverse component,
    // or in a round of their own
    constexpr int LG = G >= NI + 3 ? NI : 0;
    cplx<R> w[RI][8];
#pragma unroll
    for (int q = 0; q < RI; ++q) {
        const int c = q * G + g;
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            if (c >= NI) {
                w[q][r] = {R(0), R(0)};
                continue;
            }
            const cplx<R> p = X[c * (N + 1) + ext_pos<L>(t + r * TF)];
            w[q][r] = ext_value<R, L>((C::IT >> c) & 1, t + r * TF, p.x, p.y);
        }
    }
    Twiddles<R, L> tw;
    tw.load(a.W, t);
    const R *last = a.src + (size_t)a.nx * a.ldk;
    if (!FRONT && LG && first && g >= LG && g < LG + 3) {
        const int c = last_row_index(g - LG);
        load_pair<R, L>(last + c * cs, 0, false, (C::FT >> c) & 1, t, w[0]);
    }
#pragma unroll
    for (int q = 0; q < RI; ++q) {
        const int c = q * G + g;
        cplx<R> z[4], zn;
        __syncthreads();
        fft_core<R, L, H::PS>(w[q], buf, t, tw, z, zn);
        if (!FRONT && LG && first && g >= LG && g < LG + 3)
            last_row_keep<R, L>(a, g - LG, (C::FT >> last_row_index(g - LG)) & 1, t, z, zn);
        if (c >= NI) continue;
        R *da = a.dst + c * cs + row, *db = da + a.ldk;
        const int type = (C::IT >> c) & 1;
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            if (i == 4 && t) break;
            const int k = t + i * TF;
            const cplx<R> x = row_values<R, L>(type, k, i < 4 ? z[i < 4 ? i : 0] : zn, R(1));
            at(da, k) = x.x;
            at(db, k) = x.y;
        }
    }
    if (!first) return;
    if (FRONT) {
        last_row_front<R, N, BS>(a, seed, reinterpret_cast<R *>(X));
    } else if (!LG) {
#pragma unroll
        for (int q = 0; q < (3 + G - 1) / G; ++q) {
            const int i = q * G + g, c = last_row_index(i), type = (C::FT >> c) & 1;
            cplx<R> v[8], z[4], zn;
            load_pair<R, L>(last + c * cs, 0, false, type, t, v);
            __syncthreads();
            fft_core<R, L, H::PS>(v, buf, t, tw, z, zn);
            if (i < 3) last_row_keep<R, L>(a, i, type, t, z, zn);
        }
    }
}

// ---- host side ----

// kernels with more than 64 KB of dynamic LDS ask for it
template <typename K> static int grant_lds(qp_ctx *c, K kern, size_t lds)
{
    QP_REQUIRE(lds <= c->max_lds, QP_ERR_UNSUPPORTED, "field solve needs %zu B of LDS (limit %zu)",
               lds, c->max_lds);
    if (lds > 65536)
        QP_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)lds));
    return QP_OK;
}

template <typename R, int L, bool INV>
static int xt_launch(qp_ctx *c, const XtSet<R> &s, int nc, int types, int zero_row,
                     const BorderArgs<R> &bd)
{
    using X = XtShape<R, L>;
    auto kern = k_fft_xt<R, L, INV>;
    int rc = grant_lds(c, kern, X::LDS);
    if (rc) return rc;
    const int nrows = INV ? c->ny : c->ny + 1;
    const int groups = (nrows + X::ROWS - 1) / X::ROWS;
    const double ani = 1.0 / ((double)c->nx * (double)c->ny);
    ResJob rj{};
    if (INV) {
        rj = c->res_job;
        c->res_job = ResJob{};
    }
    {
    ProfScope _ps(c, QP_PROF_FFT, 2.0 * nc * nrows * (c->nx + 1.0) * sizeof(R));
    hipLaunchKernelGGL(kern, dim3((groups + 7) & ~7, nc), dim3(X::BS), X::LDS, c->stream, s, nrows,
                       INV ? c->ldk : c->ldr, INV ? c->ldr : c->ldk, types,
                       (R)(INV ? 2.0 : ani), c->twx.as<cplx<R>>(), INV ? c->ny : -1, zero_row,
                       c->skip, rj, bd);
    }
    QP_LAUNCH_CHECK();
    return QP_OK;
}

template <typename R, int L, bool FRONT>
static int mid_launch(qp_ctx *c, const MidArgs<R> &a)
{
    using H = MidShape<R, L>;
    auto kern = k_mid<R, L, FRONT>;
    const size_t lds = H::LDS;
    const int bs = H::BS;
    int rc = grant_lds(c, kern, lds);
    if (rc) return rc;
    {
    // two y transforms of each component and the planes of the modes
    const double planes = FRONT ? 2 * 2 + 2 * 7 + 8 : 2 * 8 + 2 * 4 + 4;
    ProfScope _ps(c, QP_PROF_KSPACE, planes * (c->nx + 1.0) * (c->ny + 1.0) * sizeof(R));
    hipLaunchKernelGGL(kern, dim3(c->nx / 2), dim3(bs), lds, c->stream, a);
    }
    QP_LAUNCH_CHECK();
    return QP_OK;
}

#define QP_BY_LENGTH(n, CALL)                                       \
    switch (n) {                                                    \
    case 16: return CALL(5);                                        \
    case 32: return CALL(6);                                        \
    case 64: return CALL(7);                                        \
    case 128: return CALL(8);                                       \
    case 256: return CALL(9);                                       \
    case 512: return CALL(10);                                      \
    case 1024: return CALL(11);                                     \
    }                                                               \
    set_error("field solve: transform length %d unsupported", n);   \
    return QP_ERR_UNSUPPORTED

template <typename R, bool INV>
static int xt(qp_ctx *c, const XtSet<R> &s, int nc, int types, int zero_row,
              const BorderArgs<R> &bd = BorderArgs<R>{})
{
#define QP_CALL(L) xt_launch<R, L, INV>(c, s, nc, types, zero_row, bd)
    if constexpr (sizeof(R) == 4)
        if (c->nx == 2048) return QP_CALL(12);
    QP_BY_LENGTH(c->nx, QP_CALL);
#undef QP_CALL
}

template <typename R, bool FRONT> static int mid(qp_ctx *c, const MidArgs<R> &a)
{
#define QP_CALL(L) mid_launch<R, L, FRONT>(c, a)
    QP_BY_LENGTH(c->ny, QP_CALL);
#undef QP_CALL
}

// Whether the slice loop's field solves run here: sizes (above), and the
// transforms' tuning knob at its default (its other values select among the
// separate transforms)
bool fused_fields(const qp_ctx *c)
{
    return c->nx <= 1024 && c->ny <= 1024 && c->max_lds >= 163840 &&
           c->tune[QP_TUNE_FFT] == tune_default_of(c->prec, QP_TUNE_FFT);
}

// whether they form the border sums of the deposits in front of them
bool fused_border(const qp_ctx *c) { return fused_fields(c) && c->nx <= BORDER_MAX; }

// x types of the components that k_mid takes and gives: the pair (x, y) of
// kind_types for cu (kind 1), dcu (1), amu (3); qb, qe (1); fxy (1), psi (1),
// psit (1), bxyz (2)
static constexpr int XF_PASS = 0x89, XI_PASS = 0xc, XF_FRONT = 0, XI_FRONT = 0x61;

template <typename R>
static int solve_t(const PassFields &f, const FrontFields *fr, double dex, int l, double tol,
                   int seed, const int *seed_hist, const BorderJob &job)
{
    qp_ctx *c = f.cu->ctx;
    const size_t rp = c->rplane, kp = c->kplane;
    R *sk = c->scr_k.as<R>(), *sr = c->scr_r.as<R>();
    XtSet<R> x{};
    int nf = 0, ni = 0;
    auto add = [&](const R **list, int &n, const qp_field2d *q) {
        for (int d = 0; d < q->dim; ++d) list[n++] = q->rs.as<R>() + d * rp;
    };
    if (fr) {
        add(x.src, nf, fr->qb);
        add(x.src, nf, fr->qe);
    } else {
        add(x.src, nf, f.cu);
        add(x.src, nf, f.dcu);
        add(x.src, nf, f.amu);
    }
    for (int i = 0; i < nf; ++i) x.dst[i] = sk + i * kp;
    // the plasma deposits leave the guard row ny folded into row 0, so zero
    // (the front's second component is the plasma's charge)
    BorderArgs<R> bd{};
    if (job.n) {
        bd.g = TileGeom{c->nx, c->ny, c->mx1, c->my1, c->ldr};
        bd.halo = static_cast<const R *>(job.halo);
        bd.halo_cs = (size_t)c->ntiles * (TILE / job.rb) * band_halo(job.rb);
        while ((1 << bd.sh) < job.rb) ++bd.sh;
        bd.fold = job.fold;
        bd.first = fr ? 1 : 0;
        bd.n = job.n;
        for (int k = 0; k < job.n; ++k) {
            bd.out.p[k] = static_cast<R *>(job.p[k]);
            bd.out.inner[k] = static_cast<const R *>(job.inner[k]);
            bd.out.outer[k] = static_cast<const R *>(job.outer[k]);
            bd.out.p2[k] = static_cast<R *>(job.p2[k]);
        }
        bd.out.scale = (R)job.scale;
        bd.out.scale2 = (R)job.scale2;
    }
    int rc = xt<R, false>(c, x, nf, fr ? XF_FRONT : XF_PASS, fr ? -1 : c->ny, bd);
    if (rc) return rc;
    MidArgs<R> a{};
    a.nx = c->nx; a.ldk = c->ldk; a.cs = kp;
    a.src = sk; a.dst = sr;
    a.W = c->twy.as<cplx<R>>();
    a.ffg = c->ffg.as<R>(); a.ffs = c->ffs.as<R>();
    a.cu = f.cu->ks.as<R>(); a.dcu = f.dcu->ks.as<R>(); a.amu = f.amu->ks.as<R>();
    a.epw = f.epw->ks.as<R>(); a.epwb = f.epwb->ks.as<R>();
    a.aa = (R)(dex * dex); a.idex = (R)(1.0 / dex); a.dex = (R)dex;
    a.partial = c->red.as<double>();
    a.flags = c->flags.as<int>();
    if (fr) {
        a.qb = fr->qb->ks.as<R>(); a.qe = fr->qe->ks.as<R>();
        a.psi = fr->psi->ks.as<R>(); a.fxy = fr->fxy->ks.as<R>();
        a.seed = seed;
        a.seed_hist = seed_hist;
        if (seed) a.ehist = fr->ehist->ks.as<R>();
        if (seed && fr->ehist2) a.ehist2 = fr->ehist2->ks.as<R>();
        rc = mid<R, true>(c, a);
    } else {
        a.skip = c->skip;
        rc = mid<R, false>(c, a);
        // the inverse x pass sums the partials (see ResJob)
        int *fl = c->flags.as<int>();
        c->res_job = ResJob{c->red.as<double>(), c->nx / 2,
                            l > 0 && l < FLAG_WORDS ? fl + l - 1 : nullptr,
                            l > 0 && l < FLAG_WORDS ? fl + l : nullptr,
                            c->h_res + (l % RES_SLOTS), c->red.as<double>() + 2 * BFQP_BLOCKS, tol};
    }
    if (rc) return rc;
    XtSet<R> y{};
    const R *outs[8] = {};
    if (fr) {
        add(outs, ni, fr->fxy);
        add(outs, ni, fr->psi);
    }
    add(outs, ni, f.psit);
    add(outs, ni, f.bxyz);
    for (int i = 0; i < ni; ++i) {
        y.src[i] = sr + i * kp;
        y.dst[i] = const_cast<R *>(outs[i]);
    }
    return xt<R, true>(c, y, ni, fr ? XI_FRONT : XI_PASS, -1);
}

// a corrector pass's field solve, from the deposited cu, dcu, amu
int fused_solve_pass(const PassFields &f, double dex, int l, double tol, const BorderJob &job)
{
    int rc = f.cu->ctx->prec == QP_FP64 ? solve_t<double>(f, nullptr, dex, l, tol, 0, nullptr, job)
                                        : solve_t<float>(f, nullptr, dex, l, tol, 0, nullptr, job);
    f.cu->state = f.dcu->state = f.amu->state = f.epw->state = 1;
    f.psit->state = f.bxyz->state = 0;
    return rc;
}

// the start of a slice, from its beam and plasma charge; seed as fused_pass
int fused_solve_front(const PassFields &f, const FrontFields &fr, double dex, int seed,
                      const int *seed_hist, const BorderJob &job)
{
    QP_REQUIRE(!seed || fr.ehist, QP_ERR_ARG, "fused_solve_front: seed without history");
    int rc = f.cu->ctx->prec == QP_FP64 ? solve_t<double>(f, &fr, dex, 0, 0.0, seed, seed_hist, job)
                                        : solve_t<float>(f, &fr, dex, 0, 0.0, seed, seed_hist, job);
    fr.qb->state = fr.qe->state = f.epwb->state = 1;
    fr.fxy->state = fr.psi->state = f.psit->state = f.bxyz->state = 0;
    return rc;
}

// the x passes of the transforms of whole fields (qp_fft.hip)
template <bool INV>
static int x_pass(qp_ctx *c, float *const *src, float *const *dst, int nc, int types)
{
    XtSet<float> s{};
    for (int i = 0; i < nc; ++i) {
        s.src[i] = src[i];
        s.dst[i] = dst[i];
    }
    return xt<float, INV>(c, s, nc, types, -1);
}
int fft_x_to_columns(qp_ctx *c, float *const *src, float *const *dst, int nc, int types)
{
    return x_pass<false>(c, src, dst, nc, types);
}
int fft_x_from_columns(qp_ctx *c, float *const *src, float *const *dst, int nc, int types)
{
    return x_pass<true>(c, src, dst, nc, types);
}

}  // namespace qp
