// The nodes on the borders of the deposits' blocks.  A deposit writes the inner
// nodes of a tile (or of a band of a tile's rows) to the plane and leaves the
// sums of its border nodes in a buffer; a border node's value is the sum over
// the blocks that meet there.  It is formed by a kernel of its own
// (k_deposit_border) or, in the slice loop, by the x transform that reads the
// plane next (k_fft_xt).
#pragma once
#include "qp_common.h"

namespace qp {

struct TileGeom {
    int nx, ny, mx1, my1, ldr;
};

// a border node's place in its block of rb rows of cells, 17 x (rb + 1) nodes
__device__ __forceinline__ int halo_index(int rb, int i, int j)
{
    if (j == 0) return i;
    if (j == rb) return 17 + i;
    if (i == 0) return 34 + (j - 1);
    return 33 + rb + (j - 1);
}

// The sum of border node (X, Y) over its blocks, in a fixed order; with fold,
// row ny is added into row 0 and cleared (PPNACGUARD2L nvp = 1).  h: the border
// buffer of one component; the blocks have rb = 2^sh rows.
template <typename R>
__device__ __forceinline__ R border_node(const TileGeom &g, const R *__restrict__ h, int sh,
                                         int fold, int X, int Y)
{
    const int rb = 1 << sh, B = TILE >> sh, myb = g.my1 * B, bsh = 4 - sh;   // B = 2^bsh
    static_assert(TILE == 16, "shifts");
    // the four blocks' values are loaded together, absent ones as any entry
    auto node_sum = [&](int XX, int YY) -> R {
        const int ty1 = YY >> sh, tx1 = XX >> 4, ly = YY & (rb - 1), lx = XX & (TILE - 1);
        const bool y0 = ty1 > 0 && ly == 0, y1 = ty1 < myb;
        const bool x0 = tx1 > 0 && lx == 0, x1 = tx1 < g.mx1;
        auto row = [&](int ty) {
            return (((ty >> bsh) * g.mx1) * B + (ty & (B - 1))) * band_halo(rb);
        };
        const int r0 = row(y0 ? ty1 - 1 : 0), r1 = row(y1 ? ty1 : 0), st = B * band_halo(rb);
        const int c0 = (x0 ? tx1 - 1 : 0) * st, c1 = (x1 ? tx1 : 0) * st;
        const R v00 = h[y0 && x0 ? r0 + c0 + halo_index(rb, TILE, rb) : 0];
        const R v01 = h[y0 && x1 ? r0 + c1 + halo_index(rb, lx, rb) : 0];
        const R v10 = h[y1 && x0 ? r1 + c0 + halo_index(rb, TILE, ly) : 0];
        const R v11 = h[y1 && x1 ? r1 + c1 + halo_index(rb, lx, ly) : 0];
        R s = R(0);
        if (y0 && x0) s += v00;
        if (y0 && x1) s += v01;
        if (y1 && x0) s += v10;
        if (y1 && x1) s += v11;
        return s;
    };
    if (fold && Y == g.ny) return R(0);
    R v = node_sum(X, Y);
    if (fold && Y == 0) v = v + node_sum(X, g.ny);
    return v;
}

// Where a deposit's node sums go.  For component c and node value v:
//   t = v (+ inner[c][node]);  t *= scale;  p[c][node] = (outer[c][node] +) t
//   p2[c][node] = v * scale2                                (when p2[c] is set)
// With null inner/outer and unit scales this is a plain overwrite; the other
// settings restate the field additions and scalings that species2d and the
// slice loop apply right after a deposit (species2d_class.f03:166-218,
// simulation_class.f03:682-685), in the same order.
template <typename R> struct DepOut {
    R *p[8];
    const R *inner[8];
    const R *outer[8];
    R *p2[8];
    R scale, scale2;
};

template <typename R>
__device__ __forceinline__ R dep_store(const DepOut<R> &o, int c, size_t idx, R v)
{
    R t = v;
    if (o.inner[c]) t = t + o.inner[c][idx];
    t = t * o.scale;
    if (o.p2[c]) o.p2[c][idx] = v * o.scale2;
    t = o.outer[c] ? o.outer[c][idx] + t : t;
    o.p[c][idx] = t;
    return t;
}

// A border sum left to the kernel that reads the planes next: planes first ..
// of its batch, whose deposit left its border nodes in halo (blocks of 2^sh rows),
// and where their values go (DepOut).  n = 0: none.
template <typename R> struct BorderArgs {
    TileGeom g;
    const R *halo;
    size_t halo_cs;
    int sh, fold, first, n;
    DepOut<R> out;
};

}  // namespace qp
