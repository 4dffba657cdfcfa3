// The slice loop's k-space arithmetic of one mode, shared by the kernels that
// run it on its own (qp_fused.hip) and between transforms (qp_spectral.hip).  The
// fused products are written out (fmadd), so that all of them give the same bits.
#pragma once

#include "qp_common.h"

namespace qp {

// One mode of PBPOISD22N_QP isign = 1 (bfqp): d1, d2 (dcu) and n1, n2 (the
// new B_perp from the old one) of mode (kx, ky); modes off the tables (tab =
// false) and (0, 0) keep dcu and get zero.  Returns whether dcu changed.
template <typename R>
__device__ __forceinline__ bool corrector_mode(bool tab, int kx, int ky, R fg, R fs, R dkx, R dky,
                                               R aa, R idex, R c3, R a1, R a2, R a3, R old1,
                                               R old2, R &d1, R &d2, R &n1, R &n2)
{
    n1 = n2 = R(0);
    if (!tab || (kx == 0 && ky == 0)) return false;
    const R at2 = R(1) * fg / fmadd(aa, fg, R(1));
    const R at1 = at2 * fs;
    const R at3 = aa * at2;
    // through values of its own: branches that store to different arguments end up
    // as one store by a selected address, and what lies there in scratch
    R s1, s2, m1 = R(0), m2 = R(0);
    if (kx > 0 && ky > 0) {
        s1 = fmadd(-dky, a3, fmadd(dkx, a1, -d1));
        const R aat1 = fmadd(-(dkx * c3), idex, s1);
        s2 = fmadd(dky, a2, fmadd(-dkx, a3, -d2));
        const R aat2 = fmadd(-(dky * c3), idex, s2);
        m1 = fmadd(at3, old1, at1 * aat1);
        m2 = fmadd(at3, old2, at1 * aat2);
    } else if (kx > 0) {
        s1 = fmadd(dkx, a1, -d1);
        s2 = fmadd(-dkx, a3, -d2);
        m2 = fmadd(at3, old2, at1 * s2);
    } else {
        s1 = fmadd(-dky, a3, -d1);
        s2 = fmadd(dky, a2, -d2);
        m1 = fmadd(at3, old1, at1 * s1);
    }
    d1 = s1;
    d2 = s2;
    n1 = m1;
    n2 = m2;
    return true;
}

// div (MPPDIVFD2) -> pot (MPPOTPD2) -> * (-dex) of the current: psit
template <typename R>
__device__ __forceinline__ R psit_mode(bool inner, R fg, R dkx, R dky, R c1, R c2, R dex)
{
    const R ps = inner ? fg * (-fmadd(dkx, c1, dky * c2)) : R(0);
    return ps * (-dex);
}

// bf (MPPBBPOISD23, ci = 1): only its z component survives the B assembly
template <typename R>
__device__ __forceinline__ R bz_mode(bool tab, int kx, int ky, R fg, R fs, R dkx, R dky, R c1, R c2)
{
    if (!tab) return R(0);
    const R at1 = R(1) * fg * fs;
    if (kx > 0 && ky > 0) return fmadd(dkx * at1, c2, -(dky * at1 * c1));
    if (kx > 0) return dkx * at1 * c2;
    if (ky > 0) return -(dky * at1) * c1;
    return R(0);
}

// The B assembly (simulation_class.f03:677-680): B_x and B_y from the corrector's
// (e1, e2) and the beam's (b1, b2)
template <typename R> __device__ __forceinline__ R bx_mode(R e2, R b2, R dex) { return fmadd(e2, -dex, -b2); }
template <typename R> __device__ __forceinline__ R by_mode(R e1, R b1, R dex) { return fmadd(e1, dex, b1); }

// The seed by extrapolation in xi of one component: e = B(j-1) becomes 2 e - h
// (seed 2) or 3 e - 3 h + g (seed 3), h = B(j-2), g = B(j-3)
template <typename R> __device__ __forceinline__ R seed_mode(int seed, R e, R h, R g)
{
    if (seed == 2) return R(2) * e - h;
    if (seed == 3) return fmadd(R(3), e, -(R(3) * h)) + g;
    return e;
}

}  // namespace qp
