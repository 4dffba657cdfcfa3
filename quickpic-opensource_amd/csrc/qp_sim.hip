// The 3-D step and its xi-slice loop on one GPU (simulation_class.f03:611-765).
//
// Field roles and states follow init_sim_fields (simulation_class.f03:267-287):
// qb, qe, psit, psi, div_vpot (1 comp), fxy, dcu, epw, epwb (2), cu, amu,
// bxyz (3); cu and epw start in k space.  Every call below enqueues on the
// context stream; the only host synchronisations are the corrector's stopping
// test (when a tolerance is given) and the particle check at the slice end.
#include <algorithm>
#include <cmath>
#include <string>
#include <thread>
#include <vector>

#include "qp_common.h"

namespace qp {
int species_push_nocheck(qp_species *sp, const qp_field2d *ef, const qp_field2d *bf,
                         const qp_field2d *psit, double dex);
int species_check(qp_species *sp);
const void *species_buffer_key(const qp_species *sp);
void species_flip(qp_species *sp, bool offsets);
int species_check_post(qp_species *sp, int slice);
void species_err_words(qp_species *sp, const int **err, int **h_err);
int species_check_mark(qp_species *sp);
int species_check_poll(qp_species *sp, bool wait);
int species_qdp_fused(qp_species *sp, qp_field2d *q, bool first, const BeamPlane *bp,
                      BorderJob *job);
int beam_slice_assign(qp_beam *b, qp_field2d *q, int slice, const int *jdev = nullptr);
int beam_slice_plane(qp_beam *b, qp_field2d *q, int slice, const int *jdev, BeamPlane *bp);
int beam_slice_add_dev(qp_beam *b, qp_field2d *q, const int *jdev);
int species_q3_initial(qp_species *sp, qp_field3d *q3);
int species_amjdp_fused(qp_species *sp, const qp_field2d *ef, const qp_field2d *bf,
                        const qp_field2d *psit, qp_field2d *cu, qp_field2d *dcu, qp_field2d *amu,
                        double dex, bool first, bool last, const qp_field2d *psi, BorderJob *job);
}  // namespace qp

struct qp_sim {
    qp_ctx *ctx;
    std::vector<qp_species *> sp;
    std::vector<qp_beam *> bm;
    std::vector<qp_field3d *> q3s;   // optional cbq targets, one per species
    qp_field3d *psi3d = nullptr;     // optional diagnostics: psi (dim 1), current (dim 3)
    qp_field3d *cu3d = nullptr;
    int iter;
    qp_field2d *f[QP_F_COUNT];
    qp_field3d *bexyz, *bbxyz;
    qp_field2d *epw_hist;   // B_perp of the slice before the last (extrapolated seed)
    qp_field2d *epw_hist2;  // and of the one before it (quadratic seed)
    qp_field2d *gprev, *fprev;   // last pass's result and change (mixed corrector)
    int hist_slices;        // slices of this step recorded in the history
    int prepared;           // slice whose first part has run (0: none)
    int last_passes;        // corrector passes of the last finished slice
    int pred_passes = 0;    // passes the next slice's corrector enqueues at once
    bool last_adaptive;     // whether its residuals were read back
    // Captured slices (qp_scan): while `graph` is set, prepare and finish
    // enqueue a slice whose index lives in device memory, so one captured
    // slice serves every j.  ctl[0] = j (the slice to run next), ctl[1] =
    // the slices recorded for the extrapolated seed; passes_dev[j] = the
    // corrector passes slice j used.  begin_step resets them.
    qp::DevBuf ctl, passes_dev;
    bool graph = false;
};

using namespace qp;

#define RC(x) do { int _r = (x); if (_r) return _r; } while (0)

namespace {

__global__ void k_ctl_reset(int *ctl)
{
    if (threadIdx.x == 0) {
        ctl[0] = 1;
        ctl[1] = 0;
    }
}

// End of a captured slice: the passes it used (pass l converged when flag
// word l is set; without a tolerance all iter_max ran), then the next slice
__global__ void k_slice_end(int *ctl, const int *flags, int iter_max, int adaptive, int seeding,
                            int *passes, int nz)
{
    if (threadIdx.x != 0) return;
    const int j = ctl[0];
    if (j < 1 || j > nz) return;
    int p = iter_max;
    if (adaptive)
        for (int l = 1; l < iter_max; ++l)
            if (flags[l]) {
                p = l;
                break;
            }
    passes[j] = p;
    ctl[0] = j + 1;
    if (seeding) ctl[1] = ctl[1] + 1;
}

}  // namespace

extern "C" {

int qp_sim_create(qp_ctx *c, qp_species *const *sp, int nsp, qp_beam *const *bm, int nb, int iter,
                  qp_sim **out)
{
    QP_REQUIRE(c && out && nsp >= 0 && nb >= 0 && iter >= 1, QP_ERR_ARG,
               "qp_sim_create: bad argument");
    qp_sim *s = new qp_sim();
    s->ctx = c;
    for (int i = 0; i < nsp; ++i) s->sp.push_back(sp[i]);
    for (int i = 0; i < nb; ++i) s->bm.push_back(bm[i]);
    s->q3s.assign(nsp, nullptr);
    s->iter = iter;
    static const int dims[QP_F_COUNT] = {1, 1, 1, 1, 1, 2, 3, 3, 2, 3, 2, 2};
    static const int st[QP_F_COUNT] = {0, 0, 0, 0, 0, 0, 0, 1, 0, 0, 1, 0};
    int rc = QP_OK;
    for (int i = 0; i < QP_F_COUNT && !rc; ++i) rc = qp_field2d_create(c, dims[i], st[i], &s->f[i]);
    if (!rc) rc = qp_field3d_create(c, 3, &s->bexyz);
    if (!rc) rc = qp_field3d_create(c, 3, &s->bbxyz);
    if (!rc) rc = qp_field2d_create(c, 2, 1, &s->epw_hist);
    if (!rc) rc = qp_field2d_create(c, 2, 1, &s->epw_hist2);
    if (!rc) rc = qp_field2d_create(c, 2, 1, &s->gprev);
    if (!rc) rc = qp_field2d_create(c, 2, 1, &s->fprev);
    if (!rc) rc = s->ctl.alloc(4 * sizeof(int));
    if (!rc) rc = s->passes_dev.alloc((size_t)(c->nz + 2) * sizeof(int));
    if (rc) { qp_sim_destroy(s); return rc; }
    *out = s;
    return QP_OK;
}

int qp_sim_destroy(qp_sim *s)
{
    if (!s) return QP_OK;
    for (int i = 0; i < QP_F_COUNT; ++i) qp_field2d_destroy(s->f[i]);
    qp_field3d_destroy(s->bexyz);
    qp_field3d_destroy(s->bbxyz);
    qp_field2d_destroy(s->epw_hist);
    qp_field2d_destroy(s->epw_hist2);
    qp_field2d_destroy(s->gprev);
    qp_field2d_destroy(s->fprev);
    if (s->ctx) (void)hipStreamSynchronize(s->ctx->stream);
    s->ctl.release();
    s->passes_dev.release();
    delete s;
    return QP_OK;
}

int qp_sim_field2d(qp_sim *s, int which, qp_field2d **out)
{
    QP_REQUIRE(s && out && which >= 0 && which < QP_F_COUNT, QP_ERR_ARG, "qp_sim_field2d: bad argument");
    *out = s->f[which];
    return QP_OK;
}

int qp_sim_field3d(qp_sim *s, qp_field3d **bexyz, qp_field3d **bbxyz)
{
    QP_REQUIRE(s, QP_ERR_ARG, "qp_sim_field3d: null sim");
    if (bexyz) *bexyz = s->bexyz;
    if (bbxyz) *bbxyz = s->bbxyz;
    return QP_OK;
}

int qp_sim_species_q3(qp_sim *s, int species, qp_field3d *q3)
{
    QP_REQUIRE(s && species >= 0 && species < (int)s->sp.size(), QP_ERR_ARG,
               "qp_sim_species_q3: bad species index");
    s->q3s[species] = q3;
    // plane 1 holds the smoothed charge of the plasma as loaded
    return q3 ? species_q3_initial(s->sp[species], q3) : QP_OK;
}

int qp_sim_diag3d(qp_sim *s, int which, qp_field3d *f3)
{
    QP_REQUIRE(s && (which == QP_DIAG_PSI || which == QP_DIAG_CU), QP_ERR_ARG,
               "qp_sim_diag3d: bad argument");
    QP_REQUIRE(!f3 || (f3->ctx == s->ctx && f3->dim == (which == QP_DIAG_PSI ? 1 : 3)),
               QP_ERR_ARG, "qp_sim_diag3d: the 3-D field must have %d component(s)",
               which == QP_DIAG_PSI ? 1 : 3);
    (which == QP_DIAG_PSI ? s->psi3d : s->cu3d) = f3;
    return QP_OK;
}

// dim planes of a 2-D field's real space into plane lpos of a 3-D field
// (the copy of cb, field2d_class.f03:538-575, whatever the field's state)
static int copy_planes(qp_ctx *c, const qp_field2d *f, qp_field3d *f3, int lpos)
{
    size_t e = c->esize, pl = c->rplane, st = (size_t)(c->nz + 1) * pl;
    for (int i = 0; i < f3->dim; ++i) {
        char *dst = (char *)f3->buf.p + ((size_t)i * st + (size_t)(lpos - 1) * pl) * e;
        const char *src = (const char *)f->rs.p + (size_t)i * pl * e;
        QP_HIP(hipMemcpyAsync(dst, src, pl * e, hipMemcpyDeviceToDevice, c->stream));
    }
    return QP_OK;
}

int qp_sim_begin_step(qp_sim *s)
{
    QP_REQUIRE(s, QP_ERR_ARG, "qp_sim_begin_step: null sim");
    qp_ctx *c = s->ctx;
    for (qp_beam *b : s->bm) RC(qp_beam_qdp(b));
    // pipeline receive on the first stage zeroes these (ufield2d_class.f03:528-531)
    qp_field2d *cu = s->f[QP_F_CU], *epw = s->f[QP_F_EPW];
    RC(launch_fill(c, cu->ks.p, cu->dim * c->kplane, 0.0));
    cu->state = 1;
    RC(launch_fill(c, epw->ks.p, epw->dim * c->kplane, 0.0));
    epw->state = 1;
    s->hist_slices = 0;
    hipLaunchKernelGGL(k_ctl_reset, dim3(1), dim3(64), 0, c->stream, s->ctl.as<int>());
    QP_LAUNCH_CHECK();
    RC(qp_field2d_as(s->f[QP_F_FXY], 0.0));
    RC(qp_field2d_as(s->f[QP_F_PSIT], 0.0));
    RC(qp_field2d_as(s->f[QP_F_BXYZ], 0.0));
    // slice-1 copies (simulation_class.f03:639-641)
    const int d12[2] = {1, 2}, d1[1] = {1}, d3[1] = {3}, d123[3] = {1, 2, 3};
    RC(qp_field2d_cb(s->f[QP_F_FXY], s->bexyz, 1, 2, d12, d12));
    RC(qp_field2d_cb(s->f[QP_F_PSIT], s->bexyz, 1, 1, d1, d3));
    RC(qp_field2d_cb(s->f[QP_F_BXYZ], s->bbxyz, 1, 3, d123, d123));
    return QP_OK;
}

// The slice follows go_simulation (simulation_class.f03:643-736) call for
// call, with these fusions (each kernel restates the calls it replaces in
// their order):
//  * the plasma deposits write the slice's q (qdp additions) and cu, dcu,
//    amu (amjdp additions and the dex scaling of :682-685) directly;
//  * pot + grad is one k-space kernel; the inverse transforms of fxy and
//    psi, of psit and bxyz, and the forward transforms of cu, dcu, amu are
//    batched;
//  * a corrector pass (bfqp, then div, pot, * -dex for psit, then bf) and
//    the B assembly that follows it (:677-680) are one k-space kernel, so the
//    inverse transform of bxyz that opens the next pass (or follows the loop)
//    runs at the end of this one, beside psit's;
//  * -fxy + B is formed where the push gathers it and, with the predictor
//    cu -= dxi dcu and the slice writes, stored at the end of the slice by one
//    kernel; the first beam's charge plane is converted beside the first
//    species' charge deposit.

// beam charge (:650-655) and plasma charge (:657-661) of slice j
static int slice_charges(qp_sim *s, int j, BorderJob *job)
{
    qp_ctx *c = s->ctx;
    QP_REQUIRE(j >= 1 && j <= c->nz, QP_ERR_ARG, "qp_slice_prepare: slice %d outside 1..%d", j,
               c->nz);
    qp_field2d *qb = s->f[QP_F_QB], *qe = s->f[QP_F_QE];
    const int nsp = (int)s->sp.size();
    // the move check of an earlier slice, if it has arrived (captured
    // slices leave the error word on the device; qp_scan_run reads it)
    if (!s->graph)
        for (qp_species *sp : s->sp) RC(species_check_poll(sp, false));
    const int *jdev = s->graph ? s->ctl.as<int>() : nullptr;
    BeamPlane bp{};
    if (s->bm.empty()) RC(qp_field2d_as(qb, 0.0));
    else if (nsp == 0) RC(beam_slice_assign(s->bm[0], qb, j + 1, jdev));
    else RC(beam_slice_plane(s->bm[0], qb, j + 1, jdev, &bp));
    if (nsp == 0) RC(qp_field2d_as(qe, 0.0));
    for (int i = 0; i < nsp; ++i)
        RC(species_qdp_fused(s->sp[i], qe, i == 0, i == 0 && bp.q3 ? &bp : nullptr,
                             i == nsp - 1 ? job : nullptr));
    for (size_t i = 1; i < s->bm.size(); ++i)
        RC(jdev ? beam_slice_add_dev(s->bm[i], qb, jdev) : qp_beam_qdpcopy(s->bm[i], qb, j + 1));
    QP_REQUIRE(qb->state == 0 && qe->state == 0, QP_ERR_STATE, "fftrk: data is in ks");
    return QP_OK;
}

// first part of a slice: beam and plasma charge, psi, E_perp, the psi
// gather (:650-670), up to the corrector seed
int qp_slice_prepare(qp_sim *s, int j)
{
    QP_REQUIRE(s, QP_ERR_ARG, "qp_slice_prepare: null sim");
    RC(slice_charges(s, j, nullptr));
    qp_field2d **F = s->f;
    qp_field2d *qb = F[QP_F_QB], *qe = F[QP_F_QE], *psi = F[QP_F_PSI], *fxy = F[QP_F_FXY];
    qp_field2d *epwb = F[QP_F_EPWB];
    // the two forward transforms are independent and run as one batch
    {
        qp_field2d *fs[2] = {qb, qe};
        const int kinds[2] = {1, 1};
        RC(fft_r2k_batch(s->ctx, fs, kinds, 2));
        qb->state = qe->state = 1;
    }
    // the beam's transverse field (:656), psi and E_perp (:662-666)
    RC(qp_field2d_elf(qb, epwb));
    RC(fused_psi_fxy(qe, psi, fxy));
    {
        qp_field2d *fs[2] = {fxy, psi};
        const int kinds[2] = {1, 1};
        RC(fft_k2r_batch(s->ctx, fs, kinds, 2));
        fxy->state = psi->state = 0;
    }
    // the species' psi gather (:667-669) runs inside the first corrector pass
    s->prepared = j;
    return QP_OK;
}

}  // extern "C"

namespace {

// The parts of a slice after its charges, enqueued in order: begin (corrector
// seed and predictor; with front also psi and E_perp, solved for together with
// the predictor's fields), pass 1, 2, ... (head and tail), and end (push and
// slice writes).  Inside captured slices (s->graph) the slice index and the
// seed's count are read from device memory.
struct SliceRun {
    qp_sim *s;
    int j, iter_max;
    double tol;
    qp_ctx *c;
    bool adaptive, mixing, fused, bordered;
    int seed = 0, tag0 = 0;
    PassFields pf, pc;
    BorderJob border;   // the last deposit's, for the solve behind it (fused_border)

    SliceRun(qp_sim *sim, int jj, int imax, double t)
        : s(sim), j(jj), iter_max(imax), tol(t), c(sim->ctx), adaptive(t > 0.0),
          // the mixed corrector (QP_TUNE_MIX) applies only to runs to a
          // tolerance outside captured slices
          mixing(t > 0.0 && !sim->graph && sim->ctx->tune[QP_TUNE_MIX] == 1),
          fused(fused_fields(sim->ctx) && !mixing), bordered(fused && fused_border(sim->ctx)),
          pf{sim->f[QP_F_CU], sim->f[QP_F_DCU], sim->f[QP_F_AMU], sim->f[QP_F_EPW],
             sim->f[QP_F_EPWB], sim->f[QP_F_PSIT], sim->f[QP_F_BXYZ], nullptr, nullptr},
          pc(pf)
    {
        if (mixing) {
            pc.gprev = s->gprev;
            pc.fprev = s->fprev;
        }
    }

    int *flags() const { return c->flags.as<int>(); }

    // predictor fields from the carried current (:671-675) and the B assembly
    int begin(bool front)
    {
        QP_REQUIRE(iter_max >= 1, QP_ERR_ARG, "qp_slice_finish: iter_max %d", iter_max);
        s->prepared = 0;
        // the extrapolated corrector seed is applied by the predictor's kernel:
        // linear (QP_TUNE_SEED = 1) or quadratic (3) in xi
        const bool quad = c->tune[QP_TUNE_SEED] == 3;
        if (adaptive && (c->tune[QP_TUNE_SEED] == 1 || quad)) {
            seed = s->hist_slices >= 3 ? 3 : (s->hist_slices >= 2 ? 2 : 1);
            ++s->hist_slices;
        }
        const int *seed_hist = s->graph && seed ? s->ctl.as<int>() + 1 : nullptr;
        qp_field2d *hist2 = quad ? s->epw_hist2 : nullptr;
        if (front) {
            const FrontFields fr{s->f[QP_F_QB], s->f[QP_F_QE], s->f[QP_F_PSI], s->f[QP_F_FXY],
                                 s->epw_hist, hist2};
            RC(fused_solve_front(pf, fr, c->dex, seed, seed_hist, border));
        } else {
            RC(fused_pass(pf, c->dex, false, 0, 0.0, seed, s->epw_hist, seed_hist, hist2));
            RC(inverse());
        }
        // launches of pass l carry tag tag0 + l, unique to this slice, so that
        // the timing of a speculative pass that returned at once is dropped
        // without touching the earlier slices' pending timings
        c->prof_epoch = (c->prof_epoch + 1) & 0xffffff;
        tag0 = c->prof_epoch << 6;
        return QP_OK;
    }

    int inverse()
    {
        qp_field2d *inv[2] = {pf.psit, pf.bxyz};
        const int kinds[2] = {1, 2};
        RC(fft_k2r_batch(c, inv, kinds, 2));
        pf.psit->state = pf.bxyz->state = 0;
        return QP_OK;
    }

    // corrector passes (:676-710): a pass is its deposits (head) and its field
    // solve (tail); with c->skip set, its kernels return at once when flag word
    // l - 1 says that an earlier pass has converged
    int head(int l)
    {
        c->prof_tag = tag0 + l;
        if (c->skip) c->skip = flags() + (l - 1);
        const int nsp = (int)s->sp.size();
        if (nsp == 0) {
            RC(qp_field2d_as(pf.cu, 0.0));
            RC(qp_field2d_as(pf.dcu, 0.0));
            RC(qp_field2d_as(pf.amu, 0.0));
        }
        // the first pass applies the species' psi gather (extpsi, :667-669)
        // to each particle just before its deposit
        for (int i = 0; i < nsp; ++i)
            RC(species_amjdp_fused(s->sp[i], s->f[QP_F_FXY], pf.bxyz, pf.psit, pf.cu, pf.dcu,
                                   pf.amu, c->dex, i == 0, i == nsp - 1,
                                   l == 1 ? s->f[QP_F_PSI] : nullptr,
                                   bordered && i == nsp - 1 ? &border : nullptr));
        c->prof_tag = 0;
        return QP_OK;
    }

    int tail(int l)
    {
        c->prof_tag = tag0 + l;
        if (c->skip) c->skip = flags() + (l - 1);
        if (fused) {
            RC(fused_solve_pass(pf, c->dex, l, tol, border));
        } else {
            qp_field2d *fwd[3] = {pf.cu, pf.dcu, pf.amu};
            const int kinds[3] = {1, 1, 3};
            RC(fft_r2k_batch(c, fwd, kinds, 3));
            pf.cu->state = pf.dcu->state = pf.amu->state = 1;
            RC(fused_pass(pc, c->dex, true, l, tol));
            if (mixing) RC(fused_mix(pc, c->dex, l, tol, l >= 2 && l < iter_max));
            RC(inverse());
        }
        c->prof_tag = 0;
        return QP_OK;
    }

    int pass(int l)
    {
        RC(head(l));
        return tail(l);
    }

    // passes l0..l1 of a captured slice
    int captured(int l0, int l1)
    {
        c->skip = adaptive ? flags() : nullptr;
        int rc = QP_OK;
        for (int l = l0; l <= l1 && !rc; ++l) rc = pass(l);
        c->skip = nullptr;
        return rc;
    }

    int end()
    {
        const bool graph = s->graph;
        // plasma push (:727-730); B is already assembled, and E_perp (:721-723)
        // is formed where it is gathered
        for (qp_species *sp : s->sp)
            RC(species_push_nocheck(sp, s->f[QP_F_FXY], pf.bxyz, pf.psit, c->dex));
        // E_perp, the predictor current (:724-726), slice j+1 of the 3-D wake
        // (:731-735) and the move checks' words
        EndFields e{s->f[QP_F_FXY], s->f[QP_F_PSI], s->bexyz, s->bbxyz, j + 1};
        e.jdev = graph ? s->ctl.as<int>() : nullptr;
        e.ctl = graph ? nullptr : s->ctl.as<int>();
        e.hist = s->hist_slices;
        e.spec = fused;
        e.slice = j;
        if (!graph)
            for (qp_species *sp : s->sp)
                if (e.nerr < 4) {
                    species_err_words(sp, &e.err[e.nerr], &e.h_err[e.nerr]);
                    ++e.nerr;
                }
        RC(fused_slice_end(pf, e));
        if (graph) {
            hipLaunchKernelGGL(k_slice_end, dim3(1), dim3(64), 0, c->stream, s->ctl.as<int>(),
                               flags(), iter_max, adaptive ? 1 : 0, seeding() ? 1 : 0,
                               s->passes_dev.as<int>(), c->nz);
            QP_LAUNCH_CHECK();
            return QP_OK;
        }
        for (size_t i = 0; i < s->sp.size(); ++i)
            RC((int)i < e.nerr ? species_check_mark(s->sp[i]) : species_check_post(s->sp[i], j));
        return QP_OK;
    }

    bool seeding() const
    {
        return adaptive && (c->tune[QP_TUNE_SEED] == 1 || c->tune[QP_TUNE_SEED] == 3);
    }
};

// what comes before SliceRun::begin, and begin (which refuses an iter_max below 1:
// the slice is left prepared then, for qp_slice_finish)
int slice_begin(SliceRun &r)
{
    if (fused_fields(r.c) && r.iter_max >= 1) {
        RC(slice_charges(r.s, r.j, fused_border(r.c) ? &r.border : nullptr));
        return r.begin(true);
    }
    RC(qp_slice_prepare(r.s, r.j));
    return r.begin(false);
}

// the passes and the end of a slice that has begun
int slice_finish(SliceRun &r, int *iters_used, double *residual)
{
    qp_sim *s = r.s;
    qp_ctx *c = r.c;
    const double tol = r.tol;
    const int j = r.j, iter_max = r.iter_max, nsp = (int)s->sp.size();
    int l = 0;
    double res = -1.0;
    if (!r.adaptive) {
        for (l = 1; l <= iter_max; ++l) RC(r.pass(l));
        l = iter_max;
    } else if (nsp == 0 || !c->tune[QP_TUNE_SPECULATE] || iter_max >= FLAG_WORDS) {
        // read each residual in turn
        for (l = 1;; ++l) {
            RC(r.pass(l));
            QP_HIP(hipStreamSynchronize(c->stream));
            res = c->h_res[l % RES_SLOTS];
            if (res < tol || l == iter_max) break;
        }
    } else {
        // The deposits of pass l+1 are enqueued before the residual of pass
        // l is read back, so the device computes them while the host waits
        // and decides; once pass l converges, flag word l is set and those
        // deposits return at once, leaving the fields and particles of the
        // converged pass.  The field solve of pass l+1 is enqueued only when
        // pass l has not converged.  With QP_TUNE_SPECULATE = 2 the first
        // wait comes only after P whole passes, P the last slice's count:
        // the passes after a converged one return at once (the skipped
        // transforms pass the converged flag on), so the host reads P
        // residuals, first pass first, after one wait instead of P.
        struct SkipGuard {
            qp_ctx *c;
            ~SkipGuard() { c->skip = nullptr; }
        } guard{c};
        c->skip = r.flags();
        const int P = c->tune[QP_TUNE_SPECULATE] == 2
                          ? std::max(1, std::min(iter_max, s->pred_passes)) : 1;
        for (int k = 1; k <= P; ++k) RC(r.pass(k));
        QP_HIP(hipEventRecord(c->pass_ev[P & 1], c->stream));
        int lo = 1;   // the first pass whose residual has not been read
        for (l = P;; ++l) {
            const bool more = l < iter_max;
            if (more) RC(r.head(l + 1));
            QP_HIP(hipEventSynchronize(c->pass_ev[l & 1]));
            // passes lo..l ran (those after a converged one returned at once
            // and left their residual slots alone): the first below tol
            int conv = 0;
            for (int k = lo; k <= l && !conv; ++k)
                if (c->h_res[k % RES_SLOTS] < tol) conv = k;
            if (conv || !more) {
                const int last = conv ? conv : l;
                res = c->h_res[last % RES_SLOTS];
                for (int k = last + 1; k <= l + (more ? 1 : 0); ++k) prof_discard(c, r.tag0 + k);
                l = last;
                break;
            }
            RC(r.tail(l + 1));
            QP_HIP(hipEventRecord(c->pass_ev[(l + 1) & 1], c->stream));
            lo = l + 1;
        }
        s->pred_passes = l;
    }
    if (l > iter_max) l = iter_max;
    // species charge diagnostic of the last pass (cbq, :692-695): it reads
    // only the species' own q and cu, which the later steps leave untouched;
    // its one product is the 3-D charge, so it runs for species that have one
    for (size_t i = 0; i < s->sp.size(); ++i)
        if (s->q3s[i]) RC(qp_species_cbq(s->sp[i], s->q3s[i], j + 1));
    // the current of the last pass, scaled by dex, into cu3d (:696-698):
    // its real-space planes are kept by the forward transform
    if (s->cu3d) RC(copy_planes(c, r.pf.cu, s->cu3d, j + 1));
    RC(r.end());
    // psi * dex^2 into psi3d (:670-671); the slice write applied the scaling
    if (s->psi3d) RC(copy_planes(c, s->f[QP_F_PSI], s->psi3d, j + 1));
    // strict move check: wait for this slice's check before returning
    if (c->tune[QP_TUNE_STRICT])
        for (qp_species *sp : s->sp) RC(species_check_poll(sp, true));
    s->last_passes = l;
    s->last_adaptive = r.adaptive;
    if (iters_used) *iters_used = l;
    if (residual) *residual = r.adaptive ? res : -1.0;
    return QP_OK;
}

}  // namespace

extern "C" {

// the rest of the slice: corrector seed, predictor, passes, push, slice writes
int qp_slice_finish(qp_sim *s, int j, int iter_max, double tol, int *iters_used, double *residual)
{
    QP_REQUIRE(s, QP_ERR_ARG, "qp_slice_finish: null sim");
    QP_REQUIRE(s->prepared == j, QP_ERR_STATE, "qp_slice_finish: slice %d was not prepared", j);
    SliceRun r(s, j, iter_max, tol);
    RC(r.begin(false));
    return slice_finish(r, iters_used, residual);
}

int qp_slice_residuals(const qp_sim *s, double *res, int max, int *n)
{
    QP_REQUIRE(s && res && n && max >= 0, QP_ERR_ARG, "qp_slice_residuals: bad argument");
    QP_REQUIRE(s->last_adaptive, QP_ERR_STATE,
               "qp_slice_residuals: the last slice ran without a tolerance");
    const int m = s->last_passes < RES_SLOTS - 1 ? s->last_passes : RES_SLOTS - 1;
    *n = m < max ? m : max;
    QP_HIP(hipStreamSynchronize(s->ctx->stream));
    for (int l = 1; l <= *n; ++l) res[l - 1] = s->ctx->h_res[l % RES_SLOTS];
    return QP_OK;
}

int qp_slice_run(qp_sim *s, int j, int iter_max, double tol, int *iters_used, double *residual)
{
    QP_REQUIRE(s, QP_ERR_ARG, "qp_slice_run: null sim");
    SliceRun r(s, j, iter_max, tol);
    RC(slice_begin(r));
    return slice_finish(r, iters_used, residual);
}

int qp_sim_push_beams(qp_sim *s)
{
    QP_REQUIRE(s, QP_ERR_ARG, "qp_sim_push_beams: null sim");
    qp_ctx *c = s->ctx;
    for (qp_species *sp : s->sp) RC(species_check_poll(sp, true));
    for (qp_beam *b : s->bm) RC(qp_beam_push(b, s->bexyz, s->bbxyz, c->dex, c->dxi));
    return QP_OK;
}

int qp_sim_renew(qp_sim *s, double snew)
{
    QP_REQUIRE(s, QP_ERR_ARG, "qp_sim_renew: null sim");
    for (size_t i = 0; i < s->sp.size(); ++i) {
        RC(qp_species_renew(s->sp[i], snew));
        if (s->q3s[i]) RC(species_q3_initial(s->sp[i], s->q3s[i]));
    }
    QP_HIP(hipStreamSynchronize(s->ctx->stream));
    return QP_OK;
}

int qp_sim_end_step(qp_sim *s, double snew)
{
    QP_REQUIRE(s, QP_ERR_ARG, "qp_sim_end_step: null sim");
    RC(qp_sim_push_beams(s));
    return qp_sim_renew(s, snew);
}

// ---- batched scan: xi slices of many instances as HIP graphs ----

// A slice of one instance, captured on the instance's own stream.  With a fixed
// number of passes it is one graph.  To a tolerance it is cut: the start with
// SCAN_FIRST passes, one graph per further pass, and the end; the host reads the
// residuals (pinned memory) and enqueues no pass after the one that converges.
//
// The plasma push moves the particles between two sets of arrays and swaps
// the host's pointers to them, which a graph cannot repeat: each instance holds
// its slice twice, captured with each buffer parity, and launches the one that
// matches where the particles are, swapping the host pointers after each
// slice as the push would.
struct ScanPart {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;   // made when it is first launched
};

struct ScanSlice {
    ScanPart start, end;             // fixed passes: the whole slice is start
    std::vector<ScanPart> pass;      // passes SCAN_FIRST + 1 ...
};

struct ScanInstance {
    qp_sim *s = nullptr;
    ScanSlice slice[2];                // per buffer parity
    const void *key0 = nullptr;        // the particle buffer of parity 0
    bool offsets = false;              // the push swaps cell offsets
    int pred = 0;                      // passes the last slice needed
    // while a run is under way
    int parity = 0, left = 0, done = 0;
};

struct qp_scan {
    std::vector<ScanInstance> inst;
    int iter_max = 0;
    double tol = 0.0;
    bool failed = false;               // a run ended with the instances at different slices
};

}  // extern "C"

// The host polls for the slowest kernels in between, giving its core to other
// threads after a look without news; after this many it asks the stream whether
// it still runs.
static constexpr int SCAN_POLLS = 1 << 14;

// Passes in the first graph.  24 slices of 12 instances on 256^2 and 512^2, 4.8
// to 5.8 passes of at most 20: one graph holding a slice of all instances with
// all 20 passes 87 ms (a pass after convergence still costs its launches), cut
// with a wait for the slowest instance in each slice 80 ms and 33 ms for freeing
// its graphs, the instances apart from each other 76 ms and 1 ms.  The number
// rests on that scan: a slice that converges sooner launches four all the same
// (they return at once).
static constexpr int SCAN_FIRST = 4;

static void part_free(ScanPart &p)
{
    if (p.exec) (void)hipGraphExecDestroy(p.exec);
    if (p.graph) (void)hipGraphDestroy(p.graph);
}

// Launches a part, made executable by its first launch: the host does it beside
// the kernels of the other instances (12 instances, all 36 graphs of each made in
// qp_scan_create: 5.4 against 1.9 ms there, and a run took no less).  An
// executable graph belongs to the device that is current when it is made, and a
// run may be a thread's that has another one: the scan's is current for it alone.
static int part_launch(ScanPart &p, const qp_sim *s)
{
    if (!p.exec) {
        const int device = s->ctx->device;
        int cur = device;
        QP_HIP(hipGetDevice(&cur));
        if (cur != device) QP_HIP(hipSetDevice(device));
        const hipError_t e = hipGraphInstantiate(&p.exec, p.graph, nullptr, nullptr, 0);
        if (cur != device) (void)hipSetDevice(cur);
        QP_HIP(e);
    }
    QP_HIP(hipGraphLaunch(p.exec, s->ctx->stream));
    return QP_OK;
}

template <typename F> static int part_capture(ScanPart &p, const qp_scan *sc, qp_sim *s, F part)
{
    QP_HIP(hipStreamBeginCapture(s->ctx->stream, hipStreamCaptureModeRelaxed));
    const int hist = s->hist_slices;   // the captured seed counts on the device
    s->graph = true;
    SliceRun r(s, 1, sc->iter_max, sc->tol);
    int rc = part(r);
    s->graph = false;
    s->prepared = 0;
    s->hist_slices = hist;
    hipError_t e = hipStreamEndCapture(s->ctx->stream, &p.graph);
    if (!rc && e != hipSuccess) rc = hip_fail(e, "hipStreamEndCapture", __FILE__, __LINE__);
    return rc;
}

static int slice_capture(ScanSlice &sl, const qp_scan *sc, qp_sim *s)
{
    const bool adaptive = sc->tol > 0.0;
    const int first = adaptive ? std::min(SCAN_FIRST, sc->iter_max) : sc->iter_max;
    RC(part_capture(sl.start, sc, s, [&](SliceRun &r) -> int {
        RC(slice_begin(r));
        RC(r.captured(1, first));
        return adaptive ? QP_OK : r.end();
    }));
    if (!adaptive) return QP_OK;
    sl.pass.resize(sc->iter_max - first);
    for (int l = first + 1; l <= sc->iter_max; ++l)
        RC(part_capture(sl.pass[l - first - 1], sc, s,
                        [&](SliceRun &r) -> int { return r.captured(l, l); }));
    return part_capture(sl.end, sc, s, [&](SliceRun &r) -> int { return r.end(); });
}

// The graph that ends a slice has been enqueued: the host's side of its push, at
// once, so that the pointers are right whatever fails next.
static void scan_pushed(ScanInstance &in)
{
    for (qp_species *sp : in.s->sp) species_flip(sp, in.offsets);
    in.parity ^= 1;
    --in.left;
}

// enqueues the start of an instance's next slice and as many passes as its last
// one needed (fixed passes: the slice).  None of its passes is in flight: the
// ones of the slice before that ran have written their residuals.
static int scan_start(qp_scan *sc, ScanInstance &in)
{
    ScanSlice &sl = in.slice[in.parity];
    if (sc->tol <= 0.0) {
        RC(part_launch(sl.start, in.s));
        scan_pushed(in);
        return QP_OK;
    }
    double none = -1.0;
    for (int l = 1; l <= sc->iter_max; ++l)
        __atomic_store(in.s->ctx->h_res + l % RES_SLOTS, &none, __ATOMIC_RELAXED);
    RC(part_launch(sl.start, in.s));
    const int first = sc->iter_max - (int)sl.pass.size();
    for (in.done = first; in.done < in.pred; ++in.done)
        RC(part_launch(sl.pass[in.done - first], in.s));
    return QP_OK;
}

// One look at an instance that runs to the tolerance: news is set when its
// enqueued passes are through, after the next pass, or the end and the start of
// the next slice, have been enqueued.
static int scan_step(qp_scan *sc, ScanInstance &in, bool *news)
{
    int conv = 0;
    for (int l = 1; l <= in.done && !conv; ++l) {
        double r;
        __atomic_load(in.s->ctx->h_res + l % RES_SLOTS, &r, __ATOMIC_RELAXED);
        if (r == -1.0) return QP_OK;
        if (r >= 0.0 && r < sc->tol) conv = l;
    }
    *news = true;
    ScanSlice &sl = in.slice[in.parity];
    if (!conv && in.done < sc->iter_max) {
        const int first = sc->iter_max - (int)sl.pass.size();
        RC(part_launch(sl.pass[in.done - first], in.s));
        ++in.done;
        return QP_OK;
    }
    in.pred = conv ? conv : in.done;
    RC(part_launch(sl.end, in.s));
    scan_pushed(in);
    return in.left ? scan_start(sc, in) : QP_OK;
}

// nslices slices of every instance, from the parity of each
static int scan_slices(qp_scan *sc, int nslices)
{
    if (sc->tol <= 0.0) {
        for (int k = 0; k < nslices; ++k)
            for (ScanInstance &in : sc->inst) RC(scan_start(sc, in));
        return QP_OK;
    }
    size_t busy = nslices ? sc->inst.size() : 0;
    if (busy)
        for (ScanInstance &in : sc->inst) RC(scan_start(sc, in));
    for (int idle = 0; busy;) {
        bool news = false;
        for (ScanInstance &in : sc->inst) {
            if (!in.left) continue;
            RC(scan_step(sc, in, &news));
            if (!in.left) --busy;
        }
        if (news) {
            idle = 0;
            continue;
        }
        std::this_thread::yield();
        if (++idle == SCAN_POLLS) {
            // a stream that failed, or ended without its residual, ends the wait
            idle = 0;
            for (ScanInstance &in : sc->inst) {
                if (!in.left) continue;
                const hipError_t e = hipStreamQuery(in.s->ctx->stream);
                if (e == hipErrorNotReady) {
                    (void)hipGetLastError();
                    continue;
                }
                QP_HIP(e);
                bool now = false;
                RC(scan_step(sc, in, &now));
                QP_REQUIRE(now, QP_ERR_STATE, "qp_scan_run: a slice ended without a residual");
                if (!in.left) --busy;
            }
        }
    }
    return QP_OK;
}

extern "C" {

int qp_scan_destroy(qp_scan *sc)
{
    if (!sc) return QP_OK;
    for (ScanInstance &in : sc->inst) {
        if (in.s) (void)hipStreamSynchronize(in.s->ctx->stream);
        for (ScanSlice &sl : in.slice) {
            part_free(sl.start);
            for (ScanPart &p : sl.pass) part_free(p);
            part_free(sl.end);
        }
    }
    delete sc;
    return QP_OK;
}

int qp_scan_create(qp_sim *const *sims, int n, int iter_max, double tol, qp_scan **out)
{
    QP_REQUIRE(sims && out && n >= 1, QP_ERR_ARG, "qp_scan_create: bad argument");
    QP_REQUIRE(iter_max >= 1 && iter_max < FLAG_WORDS, QP_ERR_ARG,
               "qp_scan_create: iter_max %d outside 1..%d", iter_max, FLAG_WORDS - 1);
    for (int i = 0; i < n; ++i) {
        qp_sim *s = sims[i];
        QP_REQUIRE(s && s->ctx, QP_ERR_ARG, "qp_scan_create: null simulation %d", i);
        QP_REQUIRE(s->ctx->device == sims[0]->ctx->device, QP_ERR_ARG,
                   "qp_scan_create: instance %d is on another device", i);
        for (int k = 0; k < i; ++k)
            QP_REQUIRE(sims[k]->ctx != s->ctx, QP_ERR_ARG,
                       "qp_scan_create: instances %d and %d share a context (stream)", k, i);
        bool diag = s->cu3d || s->psi3d;
        for (qp_field3d *q3 : s->q3s) diag = diag || q3;
        QP_REQUIRE(!diag, QP_ERR_UNSUPPORTED,
                   "qp_scan_create: instance %d has 3-D diagnostics (cbq, psi, current); "
                   "captured slices do not write them", i);
        QP_REQUIRE(!s->ctx->prof_on, QP_ERR_STATE,
                   "qp_scan_create: instance %d has kernel timing on", i);
    }
    QP_HIP(hipSetDevice(sims[0]->ctx->device));
    qp_scan *sc = new qp_scan();
    sc->inst.resize(n);
    sc->iter_max = iter_max;
    sc->tol = tol;
    int rc = QP_OK;
    for (int i = 0; i < n && !rc; ++i) {
        ScanInstance &in = sc->inst[i];
        in.s = sims[i];
        if (!in.s->sp.empty()) in.key0 = species_buffer_key(in.s->sp[0]);
        in.offsets = in.s->ctx->tune[QP_TUNE_PUSH] != 1;
        // the instance's pending work (set-up, begin_step) is not part of the graphs
        hipError_t e = hipStreamSynchronize(in.s->ctx->stream);
        if (e != hipSuccess) rc = hip_fail(e, "hipStreamSynchronize", __FILE__, __LINE__);
        // each capture swaps the host pointers once (the push's host side), so
        // after the two the host is back where it started
        if (!rc) rc = slice_capture(in.slice[0], sc, in.s);
        if (!rc) rc = slice_capture(in.slice[1], sc, in.s);
    }
    if (rc) { qp_scan_destroy(sc); return rc; }
    *out = sc;
    return QP_OK;
}

int qp_scan_run(qp_scan *sc, int nslices)
{
    QP_REQUIRE(sc && !sc->inst.empty() && nslices >= 0, QP_ERR_ARG, "qp_scan_run: bad argument");
    QP_REQUIRE(!sc->failed, QP_ERR_STATE,
               "qp_scan_run: a run before ended in an error, with the simulations at different "
               "slices; begin a step of each and create the scan again");
    // the buffer parity of every instance (they must agree: an instance
    // advanced by eager slices in between would not match the graphs)
    int parity = -1;
    for (size_t i = 0; i < sc->inst.size(); ++i) {
        const ScanInstance &in = sc->inst[i];
        if (!in.key0) continue;
        const int p = species_buffer_key(in.s->sp[0]) == in.key0 ? 0 : 1;
        QP_REQUIRE(parity < 0 || p == parity, QP_ERR_STATE,
                   "qp_scan_run: instance %zu's particles are in the other buffer", i);
        parity = p;
    }
    if (parity < 0) parity = 0;
    // the slices left in each instance's step (its device slice word)
    for (size_t i = 0; i < sc->inst.size(); ++i) {
        qp_sim *s = sc->inst[i].s;
        int j = 0;
        QP_HIP(hipMemcpyAsync(&j, s->ctl.p, sizeof(int), hipMemcpyDeviceToHost, s->ctx->stream));
        QP_HIP(hipStreamSynchronize(s->ctx->stream));
        QP_REQUIRE(j >= 1 && j + nslices - 1 <= s->ctx->nz, QP_ERR_ARG,
                   "qp_scan_run: instance %zu is at slice %d; %d more exceed its %d slices", i, j,
                   nslices, s->ctx->nz);
    }
    // the instances' streams are independent, and the library's eager calls
    // before and after order with the slices on them
    for (ScanInstance &in : sc->inst) {
        in.parity = parity;
        in.left = nslices;
    }
    int rc = scan_slices(sc, nslices);
    // nothing is left running, also after an error
    for (ScanInstance &in : sc->inst) {
        const hipError_t e = hipStreamSynchronize(in.s->ctx->stream);
        if (!rc && e != hipSuccess) rc = hip_fail(e, "hipStreamSynchronize", __FILE__, __LINE__);
    }
    sc->failed = rc != QP_OK;
    RC(rc);
    // the particle move checks of the replayed slices (PPPCHECK2L)
    for (size_t i = 0; i < sc->inst.size(); ++i)
        for (qp_species *sp : sc->inst[i].s->sp) {
            int rc = species_check(sp);
            if (rc) {
                const std::string msg = qp_last_error();
                set_error("qp_scan_run: instance %zu: %s", i, msg.c_str());
                return rc;
            }
        }
    return QP_OK;
}

int qp_scan_passes(const qp_scan *sc, int instance, int *passes, int nslices)
{
    QP_REQUIRE(sc && passes && instance >= 0 && instance < (int)sc->inst.size() && nslices >= 0,
               QP_ERR_ARG, "qp_scan_passes: bad argument");
    const qp_sim *s = sc->inst[instance].s;
    QP_REQUIRE(nslices <= s->ctx->nz, QP_ERR_ARG, "qp_scan_passes: %d slices > nz", nslices);
    std::vector<int> h((size_t)s->ctx->nz + 2);
    QP_HIP(hipMemcpyAsync(h.data(), s->passes_dev.p, h.size() * sizeof(int), hipMemcpyDeviceToHost,
                          s->ctx->stream));
    QP_HIP(hipStreamSynchronize(s->ctx->stream));
    for (int j = 1; j <= nslices; ++j) passes[j - 1] = h[j];
    return QP_OK;
}

}  // extern "C"
