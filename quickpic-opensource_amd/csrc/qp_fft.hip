// Sine / cosine transforms of field2d%fftrk / fftkr on the GPU.
//
// One-dimensional definitions on nodes f(0..n) (the reference's x and y
// passes, fft2d_lib77.f:4791-5495 and the multi-component variants):
//   S(k) = sum_{j=1}^{n-1} f(j) sin(pi j k / n),            S(0) = S(n) = 0
//   C(k) = f(0)/2 + (-1)^k f(n)/2 + sum_{j=1}^{n-1} f(j) cos(pi j k / n)
// real -> k (isign = -1): x pass times 1/(nx*ny), then y pass;
// k -> real (isign = +1): y pass times 2, x pass times 2, then the guard copy
// of fftkr (field2d_class.f03:223): row ny <- row 0.
//
// GPU method (not the reference's recursion): two rows of the same type are
// packed as the real and imaginary part of the M = 2n point odd (S) or even
// (C) extension and transformed by one complex FFT.  For the even extension
// X(k) = 2 C(k) is real; for the odd one X(k) = -2i S(k); so
//   C: Re Z = 2 C_a, Im Z = 2 C_b;   S: Re Z = 2 S_b, Im Z = -2 S_a.
// The FFT is a Stockham autosort with radix-8 butterflies held in registers
// (M/8 threads per transform, 8 points each) and one closing radix-2 or
// radix-4 pass when log2(M) is not a multiple of 3.  The first pass reads the
// extension straight from memory, the last writes the n+1 outputs straight
// to memory, and the passes between exchange through LDS; the twiddle table
// entries are fetched before the first butterfly (three per radix-8 pass,
// the other powers formed by complex products).  A batch holds up to 8 components of
// any fields (grid.y); an LDS-tiled transpose sits between the x and the y
// pass.
#include "qp_fft.h"

namespace qp {

template <typename R> struct CompSet {
    const R *src[8];
    R *dst[8];
};

// Where a row pair's transform goes
template <typename R, int L, int COL> struct RowOut {
    R *da, *db, *dg;
    size_t ld;
    R half;
    int type;
    bool hb;
    __device__ __forceinline__ RowOut(const CompSet<R> &cs, int comp, int ra, int ld_dst, int type_,
                                      bool hb_, R scale, int guard_row)
        : da(cs.dst[comp] + (COL == 2 ? (size_t)ra : (size_t)ra * ld_dst)), db(da + ld_dst),
          dg((guard_row >= 0 && ra == 0) ? cs.dst[comp] + (size_t)guard_row * ld_dst : nullptr),
          ld(ld_dst), half(scale * R(0.5)), type(type_), hb(hb_)
    {
    }
    __device__ __forceinline__ void put(int k, cplx<R> x) const
    {
        const cplx<R> o = row_values<R, L>(type, k, x, half);
        if (COL == 2) {
            R *d = da + (size_t)k * ld;
            if (hb) *reinterpret_cast<cplx<R> *>(d) = o;
            else d[0] = o.x;
        } else {
            da[k] = o.x;
            if (hb) db[k] = o.y;
            if (dg) dg[k] = o.x;
        }
    }
};

// Whether k_fft_rows writes out its passes, each of the last one's values stored as
// it comes, in place of fft_core's, which hands them back: 256^2 and 512^2 FP64 up
// to 5 % shorter, 4096^2 2 %, FP32 up to 2 %; but the 4096 points of FP64 are 2 % and
// the 8192 of FP32 40 % longer so (more registers, fewer wavefronts).
template <typename R> constexpr bool own_passes(int L) { return sizeof(R) == 8 ? L != 12 : L < 13; }

// Transform rows [0, nrows) of every component of the batch along their
// contiguous axis; row pair p of component blockIdx.y is transform p.  src
// may equal dst (a block reads its rows completely before writing).  If
// guard_row >= 0 the result of row 0 is also written to row guard_row.
// COL = 1: the transform rows are the column pairs of a row-major source
// (element e of row r at src[e * ld_src + r]); COL = 2: the results are
// written as column pairs of a row-major destination (dst[k * ld_dst + r]).
// Either way a lane moves both rows of its pair with one 2-element access,
// and block b takes pair (b mod 8) * (gridDim.x / 8) + b / 8, so the blocks
// on one XCD (dispatched round-robin by block id) share cache lines.
template <typename R, int L, int COL, int PS>
__global__ void __launch_bounds__(FftShape<L>::BS)
k_fft_rows(CompSet<R> cs, int nrows, int ld_src, int ld_dst, int types, R scale,
           const cplx<R> *__restrict__ W, int guard_row, const int *skip, ResJob rj)
{
    using S = FftShape<L, PS>;
    if (skip && *skip) {
        // a pass skipped after convergence (skip is the residual job's
        // flag_in) still passes the converged flag on to the next pass
        if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0 && rj.nblk > 0 && rj.flag_out)
            *rj.flag_out = 1;
        return;
    }
    if (blockIdx.x == 0 && blockIdx.y == 0) run_res_job(rj);
    constexpr int M = S::M, n = S::N, TF = S::TF;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const int comp = blockIdx.y;
    const int type = (types >> comp) & 1;   // 0 sine, 1 cosine
    const int f = threadIdx.x / TF, t = threadIdx.x % TF;
    const int bx = COL ? (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3) : blockIdx.x;
    const int ra = 2 * (bx * S::FB + f);
    const bool live = ra < nrows, hb = ra + 1 < nrows;
    cplx<R> *buf = reinterpret_cast<cplx<R> *>(smem_raw) + f * S::LDSM;

    // The extension straight from memory: the 16 data loads are issued first
    // and unconditionally (a missing second row re-reads the first, a block
    // past the last row reads row 0; the values are then discarded), so one
    // memory latency covers them and the twiddle loads issued after them.
    R la[8], lb[8];
    {
        const R *base = cs.src[comp];
        const R *sa = live ? base + (COL == 1 ? (size_t)ra : (size_t)ra * ld_src) : base;
        // rows are read as rows except by the column-pair reader (COL = 1)
        const R *sb = (COL != 1 && live && hb) ? sa + ld_src : sa;
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const int e = ext_pos<L>(t + r * TF);
            if (COL == 1) {
                // the pair of columns ra, ra+1 of row e (ra even, ld_src even)
                const cplx<R> p2 = *reinterpret_cast<const cplx<R> *>(sa + (size_t)e * ld_src);
                la[r] = p2.x;
                lb[r] = p2.y;
            } else {
                la[r] = sa[e];
                lb[r] = sb[e];
            }
        }
    }
    if constexpr (!own_passes<R>(L)) {
        Twiddles<R, L> tw;
        tw.load(W, t);
        cplx<R> v[8], z[4], zn;
#pragma unroll
        for (int r = 0; r < 8; ++r)
            v[r] = ext_value<R, L>(type, t + r * TF, live ? la[r] : R(0),
                                   (live && hb) ? lb[r] : R(0));
        fft_core<R, L, PS>(v, buf, t, tw, z, zn);
        if (!live) return;
        const RowOut<R, L, COL> out(cs, comp, ra, ld_dst, type, hb, scale, guard_row);
#pragma unroll
        for (int i = 0; i < 4; ++i) out.put(t + i * TF, z[i]);
        if (t == 0) out.put(n, zn);
        return;
    }
    // the twiddles of every pass after the first, as Twiddles::load
    cplx<R> tw8[S::NR8 > 1 ? 3 * (S::NR8 - 1) : 1];
#pragma unroll
    for (int p = 1; p < S::NR8; ++p) {
        const int Ns = 1 << (3 * p);
        const int e = (t & (Ns - 1)) * (M / (8 * Ns));
        tw8[3 * (p - 1)] = W[e];
        tw8[3 * (p - 1) + 1] = W[2 * e];
        tw8[3 * (p - 1) + 2] = W[4 * e];
    }
    cplx<R> twr[S::REM ? 4 : 1];
    if (S::REM == 2) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            twr[2 * s] = W[t + s * TF];
            twr[2 * s + 1] = W[2 * (t + s * TF)];
        }
    } else if (S::REM == 1) {
#pragma unroll
        for (int s = 0; s < 4; ++s) twr[s] = W[t + s * TF];
    }
    cplx<R> v[8];
#pragma unroll
    for (int r = 0; r < 8; ++r)
        v[r] = ext_value<R, L>(type, t + r * TF, live ? la[r] : R(0), (live && hb) ? lb[r] : R(0));
    dft8(v);

    const RowOut<R, L, COL> out(cs, comp, ra, ld_dst, type, hb, scale, guard_row);
    auto emit = [&](int k, cplx<R> x) {
        if (live && k <= n) out.put(k, x);
    };
    static_assert(S::NR8 > 1 || S::REM != 0, "at least two passes");
#pragma unroll
    for (int r = 0; r < 8; ++r) buf[padk<PS>(8 * t + r)] = v[r];
#pragma unroll
    for (int p = 1; p < S::NR8; ++p) {
        const int Ns = 1 << (3 * p);
        __syncthreads();
        {
            const cplx<R> w1 = tw8[3 * (p - 1)], w2 = tw8[3 * (p - 1) + 1],
                          w4 = tw8[3 * (p - 1) + 2];
            const cplx<R> w3 = cmul(w2, w1);
            // (the fused product of w7 has always been the other one in FP64)
            const cplx<R> w7 = sizeof(R) == 4 ? cmul(w3, w4) : cmul(w4, w3);
            const cplx<R> w[8] = {w1, w1, w2, w3, w4, cmul(w4, w1), cmul(w4, w2), w7};
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                v[r] = buf[padk<PS>(t + r * TF)];
                if (r) v[r] = cmul(v[r], w[r]);
            }
        }
        if (p == S::NR8 - 1 && S::REM == 0) {
            dft8<true>(v);
#pragma unroll
            for (int r = 0; r < 8; ++r) emit(t + r * TF, v[r]);
            return;
        }
        dft8(v);
        __syncthreads();
        const int base = (t / Ns) * Ns * 8 + (t & (Ns - 1));
#pragma unroll
        for (int r = 0; r < 8; ++r) buf[padk<PS>(base + r * Ns)] = v[r];
    }
    __syncthreads();
    if (S::REM == 2) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int j = t + s * TF;
            const cplx<R> w1 = twr[2 * s], w2 = twr[2 * s + 1];
            cplx<R> a0 = buf[padk<PS>(j)];
            cplx<R> a1 = cmul(buf[padk<PS>(j + M / 4)], w1);
            cplx<R> a2 = cmul(buf[padk<PS>(j + M / 2)], w2);
            cplx<R> a3 = cmul(buf[padk<PS>(j + 3 * M / 4)], cmul(w2, w1));
            dft4(a0, a1, a2, a3);
            emit(j, a0);
            emit(j + M / 4, a1);
            emit(j + M / 2, a2);
        }
    } else {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int j = t + s * TF;
            cplx<R> a0 = buf[padk<PS>(j)];
            cplx<R> a1 = cmul(buf[padk<PS>(j + M / 2)], twr[s]);
            emit(j, cadd(a0, a1));
            emit(j + M / 2, csub(a0, a1));
        }
    }
}

// dst(c)[col][row] = src(c)[row][col] for row < rows, col < cols, by TS x TS
// tiles through LDS; each of the 256 threads moves TS*TS/256 elements, all
// of its loads issued before the first LDS store
template <typename R, int TS>
__global__ void __launch_bounds__(256)
k_transpose(CompSet<R> cs, int ld_src, int ld_dst, int rows, int cols, const int *skip)
{
    constexpr int RS = 256 / TS, K = TS / RS;   // rows per sweep, sweeps
    __shared__ R tile[TS][TS + 1];
    if (skip && *skip) return;
    const int comp = blockIdx.z;
    const int c0 = blockIdx.x * TS, r0 = blockIdx.y * TS;
    const int tx = threadIdx.x % TS, ty = threadIdx.x / TS;
    const R *s = cs.src[comp];
    R *d = cs.dst[comp];
    R v[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int i = ty + k * RS, r = r0 + i, c = c0 + tx;
        v[k] = (r < rows && c < cols) ? s[(size_t)r * ld_src + c] : R(0);
    }
#pragma unroll
    for (int k = 0; k < K; ++k) tile[ty + k * RS][tx] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int i = ty + k * RS, c = c0 + i, r = r0 + tx;
        if (r < rows && c < cols) d[(size_t)c * ld_dst + r] = tile[tx][i];
    }
}

void kind_types(int kind, int dim, int *tx, int *ty)
{
    // fft2d_class.f03:121-413 and the X/Y passes of the WPPF*RM* wrappers:
    // kind 1: (S,S) | (C,S),(S,C) | (C,S),(S,C),(S,S)
    // kind 2: (C,C) | (S,C),(C,S) | (S,C),(C,S),(C,C)
    // kind 3: (S,S),(S,S),(C,C)
    static const int k1[3][3][2] = {{{0, 0}}, {{1, 0}, {0, 1}}, {{1, 0}, {0, 1}, {0, 0}}};
    static const int k2[3][3][2] = {{{1, 1}}, {{0, 1}, {1, 0}}, {{0, 1}, {1, 0}, {1, 1}}};
    static const int k3[3][2] = {{0, 0}, {0, 0}, {1, 1}};
    for (int c = 0; c < dim; ++c) {
        if (kind == 1) { tx[c] = k1[dim - 1][c][0]; ty[c] = k1[dim - 1][c][1]; }
        else if (kind == 2) { tx[c] = k2[dim - 1][c][0]; ty[c] = k2[dim - 1][c][1]; }
        else { tx[c] = k3[c][0]; ty[c] = k3[c][1]; }
    }
}

static int ilog2(int v) { int l = 0; while ((1 << l) < v) ++l; return l; }

template <typename R, int L, int COL, int PS>
static int rows_launch(qp_ctx *c, const CompSet<R> &cs, int ncomp, int nrows, int ld_src,
                       int ld_dst, int types, double scale, const cplx<R> *W, int guard_row)
{
    using S = FftShape<L, PS>;
    const size_t lds = (size_t)S::FB * S::LDSM * sizeof(cplx<R>);
    QP_REQUIRE(lds <= c->max_lds, QP_ERR_UNSUPPORTED,
               "transform of length %d needs %zu B of LDS (limit %zu)", S::N, lds, c->max_lds);
    QP_REQUIRE(!COL || guard_row < 0, QP_ERR_ARG, "column transforms take no guard row");
    auto kern = k_fft_rows<R, L, COL, PS>;
    if (lds > 65536)
        QP_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)lds));
    const int pairs = (nrows + 1) / 2;
    int gx = (pairs + S::FB - 1) / S::FB;
    if (COL) gx = (gx + 7) & ~7;   // whole rounds of the 8 XCDs
    dim3 grid(gx, ncomp);
    const ResJob rj = c->res_job;
    c->res_job = ResJob{};
    {
    ProfScope _ps(c, QP_PROF_FFT, 2.0 * ncomp * nrows * (S::N + 1.0) * sizeof(R));
    hipLaunchKernelGGL(kern, grid, dim3(S::BS), lds, c->stream, cs, nrows, ld_src, ld_dst, types,
                       (R)scale, W, guard_row, c->skip, rj);
    }
    QP_LAUNCH_CHECK();
    return QP_OK;
}

template <typename R, int COL, int PS>
static int rowfft(qp_ctx *c, const CompSet<R> &cs, int ncomp, int nrows, int n, int ld_src,
                  int ld_dst, int types, double scale, const cplx<R> *W, int guard_row)
{
    switch (ilog2(2 * n)) {
    case 5: return rows_launch<R, 5, COL, PS>(c, cs, ncomp, nrows, ld_src, ld_dst, types, scale, W, guard_row);
    case 6: return rows_launch<R, 6, COL, PS>(c, cs, ncomp, nrows, ld_src, ld_dst, types, scale, W, guard_row);
    case 7: return rows_launch<R, 7, COL, PS>(c, cs, ncomp, nrows, ld_src, ld_dst, types, scale, W, guard_row);
    case 8: return rows_launch<R, 8, COL, PS>(c, cs, ncomp, nrows, ld_src, ld_dst, types, scale, W, guard_row);
    case 9: return rows_launch<R, 9, COL, PS>(c, cs, ncomp, nrows, ld_src, ld_dst, types, scale, W, guard_row);
    case 10: return rows_launch<R, 10, COL, PS>(c, cs, ncomp, nrows, ld_src, ld_dst, types, scale, W, guard_row);
    case 11: return rows_launch<R, 11, COL, PS>(c, cs, ncomp, nrows, ld_src, ld_dst, types, scale, W, guard_row);
    case 12: return rows_launch<R, 12, COL, PS>(c, cs, ncomp, nrows, ld_src, ld_dst, types, scale, W, guard_row);
    case 13: return rows_launch<R, 13, COL, PS>(c, cs, ncomp, nrows, ld_src, ld_dst, types, scale, W, guard_row);
    }
    set_error("transform length %d unsupported", n);
    return QP_ERR_UNSUPPORTED;
}

template <typename R>
static int transpose(qp_ctx *c, const CompSet<R> &cs, int ncomp, int ld_src, int ld_dst,
                     int rows, int cols)
{
    // 64 x 64 tiles in FP32 (16 elements per thread), 32 x 32 in FP64
    constexpr int TS = sizeof(R) == 4 ? 64 : 32;
    dim3 grid((cols + TS - 1) / TS, (rows + TS - 1) / TS, ncomp);
    {
    ProfScope _ps(c, QP_PROF_TRANSPOSE, 2.0 * ncomp * (double)rows * cols * sizeof(R));
    auto kern = k_transpose<R, TS>;
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, c->stream, cs, ld_src, ld_dst, rows, cols,
                       c->skip);
    }
    QP_LAUNCH_CHECK();
    return QP_OK;
}

// the form of the separate transforms (QP_TUNE_FFT; 7: the default's)
static int fft_form(const qp_ctx *c)
{
    const int v = c->tune[QP_TUNE_FFT];
    return v == 7 ? tune_default_of(c->prec, QP_TUNE_FFT) : v;
}

// the row transforms of the transpose path; QP_TUNE_FFT values 2-4 select
// another LDS padding (one pad point per 8, 32 or 4 points)
template <typename R>
static int rowfft0(qp_ctx *c, const CompSet<R> &cs, int ncomp, int nrows, int n, int ld_src,
                   int ld_dst, int types, double scale, const cplx<R> *W, int guard_row)
{
    constexpr int PD = pad_shift<R>();
    switch (fft_form(c)) {
    case 2: return rowfft<R, 0, 3>(c, cs, ncomp, nrows, n, ld_src, ld_dst, types, scale, W, guard_row);
    case 3: return rowfft<R, 0, 5>(c, cs, ncomp, nrows, n, ld_src, ld_dst, types, scale, W, guard_row);
    case 4: return rowfft<R, 0, 2>(c, cs, ncomp, nrows, n, ld_src, ld_dst, types, scale, W, guard_row);
    default: return rowfft<R, 0, PD>(c, cs, ncomp, nrows, n, ld_src, ld_dst, types, scale, W, guard_row);
    }
}

// components of a batch of fields: plane pointers and type masks
template <typename R>
static int gather_comps(qp_field2d *const *fs, const int *kinds, int nf, R **rs, R **ks,
                        int *mx, int *my)
{
    int nc = 0;
    *mx = *my = 0;
    for (int i = 0; i < nf; ++i) {
        qp_field2d *f = fs[i];
        int tx[3], ty[3];
        kind_types(kinds[i], f->dim, tx, ty);
        for (int d = 0; d < f->dim; ++d) {
            QP_REQUIRE(nc < MAX_BATCH, QP_ERR_ARG, "transform batch exceeds %d components",
                       MAX_BATCH);
            rs[nc] = f->rs.as<R>() + d * f->ctx->rplane;
            ks[nc] = f->ks.as<R>() + d * f->ctx->kplane;
            *mx |= tx[d] << nc;
            *my |= ty[d] << nc;
            ++nc;
        }
    }
    return nc;
}

// real -> k of nc components: rs[i] (real planes, pitch ldr) to ks[i]
// (k planes, pitch ldk); sr: nc scratch planes of (ny+1) x ldr for the x
// pass; mx, my: per-component sine/cosine bit masks; W: twiddles of 2nx and
// 2ny points
template <typename R>
static int r2k_core(qp_ctx *c, R *const *rs, R *const *ks, int nc, int mx, int my, R *sr,
                    int ldr, int ldk, const cplx<R> *twx, const cplx<R> *twy)
{
    const size_t pl = (size_t)(c->ny + 1) * ldr;
    CompSet<R> a{}, b{}, y{};
    for (int i = 0; i < nc; ++i) {
        a.src[i] = rs[i];
        a.dst[i] = sr + i * pl;
        b.src[i] = a.dst[i];
        b.dst[i] = ks[i];
        y.src[i] = ks[i];
        y.dst[i] = ks[i];
    }
    const double ani = 1.0 / ((double)c->nx * (double)c->ny);
    int rc = rowfft0<R>(c, a, nc, c->ny + 1, c->nx, ldr, ldr, mx, ani, twx, -1);
    if (rc) return rc;
    // y pass straight from the column pairs of the x pass (QP_TUNE_FFT 1, or 6:
    // this direction only)
    if (fft_form(c) == 1 || fft_form(c) == 6)
        return rowfft<R, 1, pad_shift<R>()>(c, b, nc, c->nx + 1, c->ny, ldr, ldk, my, 1.0,
                                            twy, -1);
    rc = transpose<R>(c, b, nc, ldr, ldk, c->ny + 1, c->nx + 1);
    if (!rc) rc = rowfft0<R>(c, y, nc, c->nx + 1, c->ny, ldk, ldk, my, 1.0, twy, -1);
    return rc;
}

// k -> real of nc components, ks[i] to rs[i]; sk: nc scratch planes of
// (nx+1) x ldk for the y pass (unused by the column-pair form)
template <typename R>
static int k2r_core(qp_ctx *c, R *const *rs, R *const *ks, int nc, int mx, int my, R *sk,
                    int ldr, int ldk, const cplx<R> *twx, const cplx<R> *twy)
{
    const size_t pl = (size_t)(c->nx + 1) * ldk;
    CompSet<R> y{}, b{}, a{}, yc{};
    for (int i = 0; i < nc; ++i) {
        y.src[i] = ks[i];
        y.dst[i] = sk + i * pl;
        b.src[i] = y.dst[i];
        b.dst[i] = rs[i];
        a.src[i] = rs[i];
        a.dst[i] = rs[i];
        yc.src[i] = ks[i];
        yc.dst[i] = rs[i];
    }
    int rc;
    // y pass written as column pairs of rs (QP_TUNE_FFT 1, or 5: this
    // direction only)
    if (fft_form(c) == 1 || fft_form(c) == 5) {
        rc = rowfft<R, 2, pad_shift<R>()>(c, yc, nc, c->nx + 1, c->ny, ldk, ldr, my, 2.0, twy,
                                          -1);
    } else {
        rc = rowfft0<R>(c, y, nc, c->nx + 1, c->ny, ldk, ldk, my, 2.0, twy, -1);
        if (!rc) rc = transpose<R>(c, b, nc, ldk, ldr, c->nx + 1, c->ny + 1);
    }
    // rows 0..ny-1; row ny receives row 0 (guard copy, PPNCGUARD2L nvp = 1)
    if (!rc) rc = rowfft0<R>(c, a, nc, c->ny, c->nx, ldr, ldr, mx, 2.0, twx, c->ny);
    return rc;
}

// Whether the x pass reads or writes the columns that the y pass works on
// (k_fft_xt), two launches in place of three.  FP32, both directions, one and
// three components: 64 x 32 19.5 -> 13.5 us; 512^2 25.3 and 33.4 -> 21.0 and
// 25.3; 1024^2 37 and 59 -> 29 and 53; 2048^2 70.6 and 157 -> 69.6 and 151.  At nx =
// 2048 a workgroup holds 4 rows, and few rows in all wait for each other longer
// than a launch takes: 2048 x 32 23.1 and 23.9 against 26.8 and 28.0 us, x 128 26.3
// and 32.7 against 28.9 and 33.6, x 256 28.7 and 42.9 against 30.1 and 38.4.
// Longer x transforms do not fit the workgroup's LDS.  FP64's column pairs take two
// launches already (512^2 23.2 and 35.9 against 26.4 and 35.3 us so).  The
// knob's other values keep the transpose or the column pairs.  nc: components of
// the batch.
static bool x_columns(const qp_ctx *c, int nc)
{
    return c->prec == QP_FP32 && (c->nx <= 1024 || (c->nx == 2048 && nc * c->ny >= 512)) &&
           c->max_lds >= 81920 &&
           c->tune[QP_TUNE_FFT] == tune_default_of(c->prec, QP_TUNE_FFT);
}

template <typename R>
static int r2k_t(qp_ctx *c, qp_field2d *const *fs, const int *kinds, int nf)
{
    R *rs[MAX_BATCH], *ks[MAX_BATCH];
    int mx, my;
    const int nc = gather_comps<R>(fs, kinds, nf, rs, ks, &mx, &my);
    if (nc <= 0) return nc;
    if constexpr (std::is_same<R, float>::value) {
        if (x_columns(c, nc)) {
            CompSet<R> y{};
            for (int i = 0; i < nc; ++i) y.src[i] = y.dst[i] = ks[i];
            int rc = fft_x_to_columns(c, rs, ks, nc, mx);
            return rc ? rc
                      : rowfft0<R>(c, y, nc, c->nx + 1, c->ny, c->ldk, c->ldk, my, 1.0,
                                   c->twy.as<cplx<R>>(), -1);
        }
    }
    return r2k_core<R>(c, rs, ks, nc, mx, my, c->scr_r.as<R>(), c->ldr, c->ldk,
                       c->twx.as<cplx<R>>(), c->twy.as<cplx<R>>());
}

template <typename R>
static int k2r_t(qp_ctx *c, qp_field2d *const *fs, const int *kinds, int nf)
{
    R *rs[MAX_BATCH], *ks[MAX_BATCH];
    int mx, my;
    const int nc = gather_comps<R>(fs, kinds, nf, rs, ks, &mx, &my);
    if (nc <= 0) return nc;
    if constexpr (std::is_same<R, float>::value) {
        if (x_columns(c, nc)) {
            R *sk[MAX_BATCH];
            CompSet<R> y{};
            for (int i = 0; i < nc; ++i) {
                sk[i] = c->scr_k.as<R>() + i * (size_t)(c->nx + 1) * c->ldk;
                y.src[i] = ks[i];
                y.dst[i] = sk[i];
            }
            int rc = rowfft0<R>(c, y, nc, c->nx + 1, c->ny, c->ldk, c->ldk, my, 2.0,
                                c->twy.as<cplx<R>>(), -1);
            return rc ? rc : fft_x_from_columns(c, sk, rs, nc, mx);
        }
    }
    return k2r_core<R>(c, rs, ks, nc, mx, my, c->scr_k.as<R>(), c->ldr, c->ldk,
                       c->twx.as<cplx<R>>(), c->twy.as<cplx<R>>());
}

int fft_r2k_batch(qp_ctx *c, qp_field2d *const *fs, const int *kinds, int nf)
{
    return c->prec == QP_FP64 ? r2k_t<double>(c, fs, kinds, nf) : r2k_t<float>(c, fs, kinds, nf);
}

int fft_k2r_batch(qp_ctx *c, qp_field2d *const *fs, const int *kinds, int nf)
{
    return c->prec == QP_FP64 ? k2r_t<double>(c, fs, kinds, nf) : k2r_t<float>(c, fs, kinds, nf);
}

int fft_r2k(qp_field2d *f, int kind) { return fft_r2k_batch(f->ctx, &f, &kind, 1); }

int fft_k2r(qp_field2d *f, int kind) { return fft_k2r_batch(f->ctx, &f, &kind, 1); }

}  // namespace qp

