// Kernels of the learned corrector seed: a U-Net of 3x3 convolutions whose
// forward and backward passes run on the MFMA units in BF16 with FP32
// accumulation.
//
// Activations are BF16 (raw 16-bit patterns) in NHWC order with a channel
// stride, so a concatenation is two layers writing disjoint channel ranges
// of one buffer.  Weights of a 3x3 convolution are BF16 [tap][cout][cin],
// tap = 3 (dy+1) + dx + 1; biases and every gradient accumulator are FP32.
// Channel counts are multiples of 16 (the input layer is zero-padded).
//
// MFMA v_mfma_f32_16x16x16bf16_1k, one wave: lane l holds A[l%16][4(l/16)+i],
// B[4(l/16)+i][l%16] and D[4(l/16)+i][l%16], i = 0..3.
#include <algorithm>
#include <atomic>
#include <cmath>

#include "qp_common.h"
#include "../../include/qpnet.h"

namespace qp {

typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint16_t f2bf(float f)
{
    // round to nearest even (inputs are finite)
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// 4 consecutive BF16 channels as an MFMA operand (8-byte aligned)
__device__ __forceinline__ v4s frag(uint2 u)
{
    v4s r;
    r[0] = (short)(u.x & 0xffff);
    r[1] = (short)(u.x >> 16);
    r[2] = (short)(u.y & 0xffff);
    r[3] = (short)(u.y >> 16);
    return r;
}
__device__ __forceinline__ v4s load4(const uint16_t *p)
{
    return frag(*reinterpret_cast<const uint2 *>(p));
}

// ---------------------------------------------------------------------------
// 3x3 convolution, 'same' zero padding:
//   y[p][co] = bias[co] + sum_{tap, ci} x'[p + off(tap)][ci] w[tap][co][ci]
// x' = x, or x * (mask > 0) when mask is given (the ReLU derivative of the
// layer that produced x, for the data gradient).  out = relu?(y) as BF16,
// added to out when accum.
//
// A wave computes 16 pixels of one row and 16 output channels, as one chain of
// 9 cin / 16 MFMAs (tap by tap, 16 input channels at a time).  What bounds it is
// the latency of the operands, which come from the caches beyond L2 (other dies
// wrote them; the seed network's layers hold 0.1 to 2 MB), so there is a wave
// for every tile, 16 to 768 blocks a convolution of a training step at 128^2,
// and two ways of not waiting for each step:
//  k_conv3x3: the channel counts it is compiled for, up to 192 (3 x 66 pixels and
//    9 x 16 weight rows of 400 bytes, 137 KB of LDS).  A block's waves are TX x TY pixel
//    groups, and the pixels around them (zero outside the plane, masked) and the
//    weights go to LDS first, in loads of 16 bytes that are in flight together.
//    A row of LDS is a pixel or a (tap, co), padded by 16 bytes: the 16 rows of
//    an operand then lie in different banks.
//  k_conv3x3_deep: others, operands not aligned to 16 bytes, and devices whose
//    workgroups have less LDS than a layer asks for.  The chain is cut in groups of
//    9 steps, whose loads are issued before the group in front is multiplied.
//  k_conv3x3_wide: those where the plane alone fills the device with waves, and
//    masked layers of few input and many output channels there.  A wave
//    computes all output channels of its pixels, step by step, and reads them once
//    in place of once for every 16 output channels.
// All by k_conv3x3_wide took 33.7 us a convolution (27 of a training step), by
// k_conv3x3_deep 11.8 us, by k_conv3x3 5.7 us (8.2 us with the channel count as an
// argument: a wave alone on its SIMD then waited for the scalar address arithmetic
// of each step).
// ---------------------------------------------------------------------------
// D[pixel 4q+i][co]: pixels xp.. of row y
__device__ __forceinline__ void conv_store(v4f acc, const float *bias, int co, int y, int xp, int W,
                                           uint16_t *out, int cs_out, int relu, int accum)
{
    const float bv = bias ? bias[co] : 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (xp + i >= W) continue;
        float v = acc[i] + bv;
        if (relu) v = v > 0.f ? v : 0.f;
        uint16_t *o = out + ((size_t)y * W + xp + i) * cs_out + co;
        if (accum) v += bf2f(*o);
        *o = f2bf(v);
    }
}

// quotient of small numbers, 0 <= a < 2^20, 1 <= b: ib = 1 / b
__device__ __forceinline__ int small_div(int a, float ib) { return (int)(((float)a + 0.5f) * ib); }

__device__ __forceinline__ uint32_t positive2(uint32_t v, uint32_t k)
{
    const bool lo = bf2f((uint16_t)k) > 0.f, hi = bf2f((uint16_t)(k >> 16)) > 0.f;
    return (lo ? v & 0xffffu : 0u) | (hi ? v & 0xffff0000u : 0u);
}

template <int KT, bool MASK>   // 16 KT input channels
__global__ void __launch_bounds__(256)
k_conv3x3(const uint16_t *__restrict__ x, const uint16_t *__restrict__ mask, int H, int W, int nbx,
          int tx, int ty, int cs_in, const uint16_t *__restrict__ w,
          const float *__restrict__ bias, uint16_t *out, int cs_out, int Cout, int relu, int accum)
{
    extern __shared__ uint4 lds4[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int by = blockIdx.x / nbx, bx = blockIdx.x - by * nbx;
    const int x0 = bx * 16 * tx, y0 = by * ty;        // the block's first pixel
    const int rw = 16 * tx + 2, npx = rw * (ty + 2);  // the pixels around it
    constexpr int Cin = 16 * KT, kc = Cin >> 3, ld = kc + 1;   // 16-byte words of a row, pitch
    const float irw = 1.f / (float)rw;
    // thread: word c of the rows r, r + rs, ...; a few threads are left over
    constexpr int rs = 256 / kc;
    const int r = tid / kc, c = tid - r * kc;
    const int cot = blockIdx.y;
    const uint16_t *wc = w + ((size_t)16 * cot * Cin + 8 * c);
    // rows y0 - 1 ..: offsets from here are small; outside the plane the block's
    // first pixel is read, and its value is dropped
    const size_t orow = (size_t)y0 * W * cs_in + 8 * c;
    const uint16_t *xc = x + orow, *kc0 = mask + (MASK ? orow : 0);
    constexpr int UW = 9, UP = 10;
    for (int w0 = r, p0 = r; r < rs && (w0 < 144 || p0 < npx); w0 += UW * rs, p0 += UP * rs) {
        uint4 vw[UW], vp[UP], vk[MASK ? UP : 1];
        uint32_t in = 0;   // bit u: inside the plane
#pragma unroll
        for (int u = 0; u < UW; ++u) {
            const int row = min(w0 + u * rs, 143);
            vw[u] = *reinterpret_cast<const uint4 *>(
                wc + (uint32_t)(((row >> 4) * Cout + (row & 15)) * Cin));
        }
#pragma unroll
        for (int u = 0; u < UP; ++u) {
            const int row = min(p0 + u * rs, npx - 1);
            const int ry = small_div(row, irw), rx = row - ry * rw;
            const int yy = y0 + ry - 1, xx = x0 + rx - 1;
            const bool ok = (unsigned)yy < (unsigned)H && (unsigned)xx < (unsigned)W;
            const ptrdiff_t o = ok ? ((ry - 1) * W + xx) * cs_in : x0 * cs_in;
            vp[u] = *reinterpret_cast<const uint4 *>(xc + o);
            if (MASK) vk[u] = *reinterpret_cast<const uint4 *>(kc0 + o);
            in |= (uint32_t)ok << u;
        }
#pragma unroll
        for (int u = 0; u < UW; ++u)
            if (w0 + u * rs < 144) lds4[(npx + w0 + u * rs) * ld + c] = vw[u];
#pragma unroll
        for (int u = 0; u < UP; ++u) {
            uint4 q = vp[u];
            if (MASK)
                q = uint4{positive2(q.x, vk[u].x), positive2(q.y, vk[u].y),
                          positive2(q.z, vk[u].z), positive2(q.w, vk[u].w)};
            if (!((in >> u) & 1)) q = uint4{0, 0, 0, 0};
            if (p0 + u * rs < npx) lds4[(p0 + u * rs) * ld + c] = q;
        }
    }
    __syncthreads();
    const int wy = wave / tx, y = y0 + wy, px0 = x0 + 16 * (wave - wy * tx);
    if (wy >= ty || y >= H || px0 >= W) return;
    const int m = lane & 15, q = lane >> 4;           // A row (pixel) and k quad
    const uint2 *l2 = reinterpret_cast<const uint2 *>(lds4);
    constexpr int ld2 = 2 * ld;
    const uint2 *pa = l2 + (wy * rw + 16 * (wave - wy * tx) + m) * ld2 + q;
    const uint2 *pb = l2 + (npx + m) * ld2 + q;
    // a tap's operands are read while the tap before is multiplied
    uint2 fa[2][KT], fb[2][KT];
    auto load = [&](int tap, uint2 *a, uint2 *b) {
        const uint2 *ta = pa + (tap / 3 * rw + tap % 3) * ld2, *tb = pb + 16 * tap * ld2;
#pragma unroll
        for (int k = 0; k < KT; ++k) {
            a[k] = ta[4 * k];
            b[k] = tb[4 * k];
        }
    };
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    load(0, fa[0], fb[0]);
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) {
        if (tap < 8) load(tap + 1, fa[(tap + 1) & 1], fb[(tap + 1) & 1]);
#pragma unroll
        for (int k = 0; k < KT; ++k)
            acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(frag(fa[tap & 1][k]),
                                                            frag(fb[tap & 1][k]), acc, 0, 0, 0);
    }
    conv_store(acc, bias, 16 * cot + m, y, px0 + 4 * q, W, out, cs_out, relu, accum);
}

template <bool MASK> struct ConvFrag {
    v4s a[9], b[9], k[MASK ? 9 : 1];
    uint32_t in;   // bit i: step i's pixel is inside
};

template <bool MASK>
__global__ void __launch_bounds__(256)
k_conv3x3_deep(const uint16_t *__restrict__ x, const uint16_t *__restrict__ mask, int H, int W, int gw,
          int cs_in, int Cin, const uint16_t *__restrict__ w, const float *__restrict__ bias,
          uint16_t *out, int cs_out, int Cout, int relu, int accum)
{
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = blockIdx.x * 4 + wave;              // this wave's pixel group
    if (g >= H * gw) return;
    const int y = g / gw, px0 = (g - y * gw) * 16;
    const int m = lane & 15, q = lane >> 4;           // A row (pixel) and k quad
    const int co = 16 * blockIdx.y + m;
    const int KT = Cin >> 4;
    const uint16_t *wl = w + (size_t)co * Cin + 4 * q;
    int tap = 0, c = 0;                               // of the next step to load
    auto load = [&](ConvFrag<MASK> &f) {
        f.in = 0;
#pragma unroll
        for (int i = 0; i < 9; ++i) {
            const int ty = (tap * 11) >> 5;           // tap / 3
            const int yy = y + ty - 1, xx = px0 + m + (tap - 3 * ty) - 1;
            const bool in = yy >= 0 && yy < H && xx >= 0 && xx < W;
            // outside: any address of the plane, the value is dropped
            const size_t o = (size_t)(in ? yy : 0) * W * cs_in + (in ? xx : 0) * cs_in + 16 * c + 4 * q;
            f.in |= (uint32_t)in << i;
            f.a[i] = load4(x + o);
            if (MASK) f.k[i] = load4(mask + o);
            f.b[i] = load4(wl + (size_t)tap * Cout * Cin + 16 * c);
            if (++c == KT) { c = 0; ++tap; }
        }
    };
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const ConvFrag<MASK> &f) {
#pragma unroll
        for (int i = 0; i < 9; ++i) {
            v4s a = f.a[i];
            const bool in = (f.in >> i) & 1;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (!in) a[j] = 0;
                if (MASK)
                    if (!(bf2f((uint16_t)f.k[i][j]) > 0.f)) a[j] = 0;
            }
            acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, f.b[i], acc, 0, 0, 0);
        }
    };
    ConvFrag<MASK> f0, f1;
    if (KT > 0) load(f0);
    for (int k = 0; k < KT; k += 2) {
        if (k + 1 < KT) load(f1);
        multiply(f0);
        if (k + 1 >= KT) break;
        if (k + 2 < KT) load(f0);
        multiply(f1);
    }
    conv_store(acc, bias, co, y, px0 + 4 * q, W, out, cs_out, relu, accum);
}

constexpr int MAXNT = 12;   // 192 output channels

__global__ void __launch_bounds__(256)
k_conv3x3_wide(const uint16_t *__restrict__ x, const uint16_t *__restrict__ mask, int H, int W,
               int gw, int cs_in, int Cin, const uint16_t *__restrict__ w,
               const float *__restrict__ bias, uint16_t *out, int cs_out, int Cout, int relu,
               int accum)
{
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = blockIdx.x * 4 + wave;              // this wave's pixel group
    if (g >= H * gw) return;
    const int y = g / gw, px0 = (g - y * gw) * 16;
    const int m = lane & 15, q = lane >> 4;           // A row (pixel) and k quad
    const int NT = Cout >> 4;
    v4f acc[MAXNT];
#pragma unroll
    for (int t = 0; t < MAXNT; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
    for (int tap = 0; tap < 9; ++tap) {
        const int yy = y + tap / 3 - 1, xx = px0 + m + tap % 3 - 1;
        const bool in = yy >= 0 && yy < H && xx >= 0 && xx < W;
        const size_t pix = in ? ((size_t)yy * W + xx) * cs_in : 0;
        for (int c0 = 0; c0 < Cin; c0 += 16) {
            v4s a = {0, 0, 0, 0};
            if (in) {
                a = load4(x + pix + c0 + 4 * q);
                if (mask) {
                    const v4s mk = load4(mask + pix + c0 + 4 * q);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (!(bf2f((uint16_t)mk[i]) > 0.f)) a[i] = 0;
                }
            }
            const uint16_t *wt = w + ((size_t)tap * Cout + m) * Cin + c0 + 4 * q;
#pragma unroll
            for (int t = 0; t < MAXNT; ++t)
                if (t < NT)
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
                        a, load4(wt + (size_t)t * 16 * Cin), acc[t], 0, 0, 0);
        }
    }
#pragma unroll
    for (int t = 0; t < MAXNT; ++t)
        if (t < NT)
            conv_store(acc[t], bias, 16 * t + m, y, px0 + 4 * q, W, out, cs_out, relu, accum);
}

// Whether k_conv3x3_wide takes a layer that k_conv3x3 does not: from this many
// pixel groups a compute unit on.  Ratio of k_conv3x3_wide's time to
// k_conv3x3_deep's on 128^2 (4 groups a unit), 160^2 (6), 192^2 (9), 224^2 (12) and
// 256^2 (16): 80 -> 192 channels 1.43, 0.96, 0.83, 0.75, 0.65; 80 -> 48 1.49, 1.13,
// 1.03, 0.87, 0.74; 256 -> 96 0.72 .. 0.59; 256 -> 32 1.07, 0.80, 0.90, 0.86, 0.75;
// 64 -> 96, not aligned, 1.13, 1.08, 1.10, 1.08, 0.86; 16 output channels 1.0 at most.
static bool conv_wide(int cus, long long groups, int cin, int cout)
{
    if (cout < 32) return false;
    const int need = cin < 80 ? 14 : cin <= 208 ? (cout >= 96 ? 6 : 10) : (cout >= 48 ? 4 : 6);
    return groups >= (long long)need * cus;
}

// And whether a masked one that k_conv3x3 has: it reads pixels and mask once for
// every 16 output channels, which with up to 48 input channels is what its time goes
// to.  Ratio of k_conv3x3_wide's time to k_conv3x3's at 160^2, 192^2, 224^2, 256^2 and
// 1024^2: 16 -> 32 channels 1.11, 1.04, 0.92, 0.86, 0.83; 16 -> 64 0.91, 0.85, 0.69,
// 0.63, 0.57; 16 -> 192 0.74, 0.67, 0.48, 0.51, 0.41 (1150 -> 477 us); 48 -> 64 1.37
// .. 1.01, 1.08; 48 -> 96 1.26, 1.22, 1.02, 0.90, 0.95; 48 -> 192 1.35, 1.19, 0.91,
// 0.87, 0.84; 32 -> 192 1.06, 1.16, 0.98, 0.90, 0.84; 64 -> 192 2.5 at least;
// 16 -> 192 without a mask 1.44 .. 1.07, 0.94.
static bool conv_wide_masked(int cus, long long groups, int cin, int cout)
{
    if (cin > 48 || cout < (cin == 16 ? 32 : 96)) return false;
    const int need = cin == 16 ? (cout >= 64 ? 6 : cout >= 48 ? 9 : 12)
                     : cin == 48 && cout >= 128 ? 12 : 16;
    return groups >= (long long)need * cus;
}

// ---------------------------------------------------------------------------
// Tables of a launch over several layers: block b belongs to the entry e with
// first[e] <= b < first[e + 1].  A table is read in the kernel's argument
// segment.
// ---------------------------------------------------------------------------
constexpr int MAXL = 16;   // convolutions of one launch
constexpr int MAXE = 36;   // vectors of one launch

__device__ __forceinline__ int table_entry(const int *first, int n)
{
    const int lane = threadIdx.x & 63;
    const bool behind = lane < n && first[lane < n ? lane : 0] <= (int)blockIdx.x;
    return (int)__popcll(__ballot(behind)) - 1;
}

// ---------------------------------------------------------------------------
// Weight and bias gradients of 3x3 convolutions:
//   dw[tap][co][ci] = sum_p dy'[p][co] x[p + off(tap)][ci]
//   db[co]          = sum_p dy'[p][co]
// dy' = dy * (yout > 0) (ReLU derivative from the layer's own output).  The
// reduction over pixels is the MFMA K dimension (db: against ones).  The pixels
// are cut in nchunk chunks, a chunk in four interleaved runs of 16-pixel
// groups; a run is one MFMA chain, its chunk's four are added in order, and so
// are the chunks.
//
// A wave takes a chunk for one (co tile, ci tile, row of taps): the three taps
// of a row share dy' and six pixels of x, 14 loads a step of three MFMAs, and
// its four runs are four independent steps, so 56 loads are in flight.  A block
// has four waves.  Chunks of at most WG_WHOLE pixels: a block goes through all
// chunks, 16 at a time, and adds them up in LDS.  Larger ones: four chunks a
// block, or one where waves are few (wgrad_few), and k_sum_parts adds the partial
// sums from memory.  All layers of a
// network go in one launch: at 128^2 a block per (tile, tap, chunk), a serial
// sum for db and two sums over the chunks, layer by layer, took 68 us a layer;
// the 14 layers together take 41 us and the sum 4 us.
// ---------------------------------------------------------------------------
constexpr int WG_WHOLE = 64;   // one step of the four runs
constexpr int WG_SLOTS = 16;
// Up to this many waves a compute unit (of a launch's layers together) the four
// runs of a chunk of `per` pixels go to four waves, four steps of one run at once,
// with the same sums in the same order: a wave's loads wait for each other's, and
// with few waves nothing else runs.  A chunk of few steps leaves such waves without
// pixels.  us, a chunk a wave against four, 32 chunks of 128, 192, 256, 512, 1024 and
// 4096 pixels: 16 -> 16 channels (0.4 waves) 12.5 and 12.2, 14.0 and 12.0, 16.1 and
// 12.1, 25.4 and 12.1, 43 and 17, 151 and 46; 48 -> 48 (3.4) 13.1 and 14.3, 15.0 and
// 14.0, 17.6 and 14.5, 26 and 19, 44 and 30, 153 and 91; 128 -> 64 (12) 19 and 27,
// 22 and 28, 26 and 28, 39 and 41, 66 and 66, 227 and 224; 512^2 96 -> 96 (13.5, 8192
// pixels) 654 and 530; 300^2 64 -> 192 (18, 2813) 276 and 276; 1024^2 16 -> 16, one
// chunk: 38.6 and 10.5 ms.
static int wgrad_few(int per) { return per >= 768 ? 16 : per >= 192 ? 4 : 0; }

struct WgradLayer {
    const uint16_t *x, *dy, *yout;
    float *dw, *db;        // db may be null
    float *part, *partb;   // partial sums per chunk (part null: of the bias alone)
    int cs_in, cin, cs_out, cout, H, W;
    int mode;              // WG_*
};
// a block takes: all chunks, and adds them up; four chunks, one a wave; one chunk,
// a run of it a wave
constexpr int WG_ALL = 0, WG_FOUR = 1, WG_ONE = 2;
struct WgradArgs {
    WgradLayer l[MAXL];
    int first[MAXL];
    int n, nchunk;
};

struct WgradTile {
    v4f w[3], b;   // taps (dyo, -1..1) and the bias: D[co 4q + i][ci m]
};

// NC chunks at once, each in its first 4 / NC runs (the others have no pixels: a
// chunk of at most 16 pixels has one run).  A chunk's tile is r[4 / NC * chunk].
// NC = 0: run `run` of one chunk alone, four of its steps at once; its tile is r[0].
template <int NC>
__device__ __forceinline__ void wgrad_runs(const WgradLayer &L, int co, int ci, int dyo, bool bias,
                                           const int *p0, const int *p1, int q, WgradTile *r,
                                           int run = 0)
{
    constexpr int NV = NC ? 4 / (NC ? NC : 1) : 4;
    constexpr int STEP = NC ? 64 : 256;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
#pragma unroll
        for (int t = 0; t < 3; ++t) r[v].w[t] = v4f{0.f, 0.f, 0.f, 0.f};
        r[v].b = v4f{0.f, 0.f, 0.f, 0.f};
    }
    const int H = L.H, W = L.W, npix = H * W;
    const v4s one = {(short)0x3f80, (short)0x3f80, (short)0x3f80, (short)0x3f80};
    const bool small = npix < (1 << 20);
    const float iw = 1.f / (float)W;
    for (int g = 0; g < (NC > 1 ? min(npix, 64) : p1[0] - p0[0]); g += STEP) {
        uint16_t d[4][4], yo[4][4], xv[4][6];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            // pixel p of the plane is p - g0 elements of cs on from the bases; a
            // pixel's neighbour (dyo, dx) is dyo W + dx pixels on; past the plane's
            // ends the last or first pixel stands in, and is dropped below
            const int g0 = min(p0[v / NV] + g + (NC ? 0 : 64 * v), npix - 1);
            const uint16_t *dyp = L.dy + (size_t)g0 * L.cs_out, *yp = L.yout + (size_t)g0 * L.cs_out;
            const uint16_t *xp = L.x + ((ptrdiff_t)g0 - W - 1) * L.cs_in;
            const int dmax = min(npix - 1 - g0, 63);
            const int xlo = max(0, W + 1 - g0), xhi = min(npix - 1 - g0, 64 + 2 * W) + W + 1;
            const int p = 16 * (NC ? v % NV : run) + 4 * q;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t o = (uint32_t)__mul24(min(p + i, dmax), L.cs_out) + co;
                d[v][i] = dyp[o];
                yo[v][i] = yp[o];
            }
#pragma unroll
            for (int j = 0; j < 6; ++j) {
                const int k = p + (dyo + 1) * W + j;
                xv[v][j] = xp[(uint32_t)__mul24(min(max(k, xlo), xhi), L.cs_in) + ci];
            }
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int p = p0[v / NV] + g + (NC ? 16 * (v % NV) : 64 * v + 16 * run) + 4 * q;
            WgradTile &s = r[NC ? v : 0];
            int py = small ? small_div(p, iw) : p / W, px = p - py * W;
            v4s a, b[3];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const bool in = p + i < p1[v / NV];
                a[i] = in && bf2f(yo[v][i]) > 0.f ? (short)d[v][i] : (short)0;
                const bool row = in && (unsigned)(py + dyo) < (unsigned)H;
                b[0][i] = row && px > 0 ? (short)xv[v][i] : (short)0;
                b[1][i] = row ? (short)xv[v][i + 1] : (short)0;
                b[2][i] = row && px + 1 < W ? (short)xv[v][i + 2] : (short)0;
                if (++px == W) { px = 0; ++py; }
            }
#pragma unroll
            for (int t = 0; t < 3; ++t)
                s.w[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b[t], s.w[t], 0, 0, 0);
            if (bias) s.b = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, one, s.b, 0, 0, 0);
        }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        if (v % NV == 0 || !NC) continue;
#pragma unroll
        for (int t = 0; t < 3; ++t) r[v - v % NV].w[t] += r[v].w[t];
        r[v - v % NV].b += r[v].b;
    }
}

// a block's chunks base .. base + ns, tiles to LDS, NC chunks of a wave at a time
template <int NC>
__device__ __forceinline__ void wgrad_slots(const WgradLayer &L, int co, int ci, int dyo, bool bias,
                                            int base, int ns, int per, int wave, int lane,
                                            v4f (*red)[3][64], float (*redb)[16])
{
    const int npix = L.H * L.W;
    for (int k0 = wave; k0 < ns; k0 += 4 * NC) {
        int p0[NC], p1[NC];
#pragma unroll
        for (int n = 0; n < NC; ++n) {
            const int k = k0 + 4 * n;
            p0[n] = k < ns ? min((base + k) * per, npix) : npix;
            p1[n] = min(npix, p0[n] + per);
        }
        WgradTile r[4];
        wgrad_runs<NC>(L, co, ci, dyo, bias, p0, p1, lane >> 4, r);
#pragma unroll
        for (int n = 0; n < NC; ++n) {
            const int k = k0 + 4 * n;
            if (k >= ns) break;
            const WgradTile &s = r[n * (4 / NC)];
#pragma unroll
            for (int t = 0; t < 3; ++t) red[k][t][lane] = s.w[t];
            if ((lane & 15) == 0) {
#pragma unroll
                for (int i = 0; i < 4; ++i) redb[k][4 * (lane >> 4) + i] = s.b[i];
            }
        }
    }
}

__global__ void __launch_bounds__(256, 3) k_wgrad(const WgradArgs A)
{
    __shared__ v4f red[WG_SLOTS][3][64];
    __shared__ float redb[WG_SLOTS][16];
    const int e = table_entry(A.first, A.n);
    const WgradLayer L = A.l[e];
    const int nchunk = A.nchunk;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m = lane & 15, q = lane >> 4;
    const int nb = L.mode == WG_ALL ? 1 : L.mode == WG_FOUR ? (nchunk + 3) / 4 : nchunk;
    const int unit = ((int)blockIdx.x - A.first[e]) / nb;
    const int cb = ((int)blockIdx.x - A.first[e]) - unit * nb;
    const int ntc = L.cin >> 4;
    const int ty = unit % 3, cit = (unit / 3) % ntc, cot = unit / 3 / ntc;
    const bool bias = L.db && cit == 0 && ty == 1;
    const int npix = L.H * L.W, per = (npix + nchunk - 1) / nchunk;
    const int tid = threadIdx.x;
    if (L.mode != WG_ALL && !L.part && !bias) return;
    if (L.mode == WG_FOUR) {
        const int chunk = cb * 4 + wave;
        if (chunk >= nchunk) return;
        const int p0 = min(chunk * per, npix), p1 = min(npix, p0 + per);
        WgradTile r[4];
        wgrad_runs<1>(L, cot * 16 + m, cit * 16 + m, ty - 1, bias, &p0, &p1, q, r);
        const WgradTile &s = r[0];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int co = cot * 16 + 4 * q + i;
#pragma unroll
            for (int t = 0; t < 3; ++t)
                if (L.part)
                    L.part[(((size_t)chunk * 9 + 3 * ty + t) * L.cout + co) * L.cin + cit * 16 +
                           m] = s.w[t][i];
            if (bias && m == 0) L.partb[(size_t)chunk * L.cout + co] = s.b[i];
        }
        return;
    }
    // where element tid of a tile belongs
    const int tl = tid >> 2, tco = cot * 16 + 4 * (tl >> 4) + (tid & 3), tci = cit * 16 + (tl & 15);
    if (L.mode == WG_ONE) {
        const int p0 = min(cb * per, npix), p1 = min(npix, p0 + per);
        WgradTile r[4];
        wgrad_runs<0>(L, cot * 16 + m, cit * 16 + m, ty - 1, bias, &p0, &p1, q, r, wave);
#pragma unroll
        for (int t = 0; t < 3; ++t) red[wave][t][lane] = r[0].w[t];
        if (m == 0)
#pragma unroll
            for (int i = 0; i < 4; ++i) redb[wave][4 * q + i] = r[0].b[i];
        __syncthreads();
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            float v = reinterpret_cast<const float *>(red[0][t])[tid];
#pragma unroll
            for (int k = 1; k < 4; ++k) v += reinterpret_cast<const float *>(red[k][t])[tid];
            if (L.part)
                L.part[(((size_t)cb * 9 + 3 * ty + t) * L.cout + tco) * L.cin + tci] = v;
        }
        if (bias && tid < 16)
            L.partb[(size_t)cb * L.cout + cot * 16 + tid] =
                ((redb[0][tid] + redb[1][tid]) + redb[2][tid]) + redb[3][tid];
        return;
    }
    // thread t sums element t of the tiles, in the order of the chunks
    float tot[3] = {0.f, 0.f, 0.f}, totb = 0.f;
    for (int base = 0; base < nchunk; base += WG_SLOTS) {
        const int ns = min(WG_SLOTS, nchunk - base);
        const int co = cot * 16 + m, ci = cit * 16 + m;
        if (per <= 16)
            wgrad_slots<4>(L, co, ci, ty - 1, bias, base, ns, per, wave, lane, red, redb);
        else if (per <= 32)
            wgrad_slots<2>(L, co, ci, ty - 1, bias, base, ns, per, wave, lane, red, redb);
        else
            wgrad_slots<1>(L, co, ci, ty - 1, bias, base, ns, per, wave, lane, red, redb);
        __syncthreads();
        for (int k = 0; k < ns; ++k) {
#pragma unroll
            for (int t = 0; t < 3; ++t) tot[t] += reinterpret_cast<const float *>(red[k][t])[tid];
            if (tid < 16) totb += redb[k][tid];
        }
        __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < 3; ++t)
        L.dw[((size_t)(3 * ty + t) * L.cout + tco) * L.cin + tci] = tot[t];
    if (bias && tid < 16) L.db[cot * 16 + tid] = totb;
}

// out[i] = sum over chunks (in order) of part[chunk][i]
struct SumArgs {
    const float *part[MAXE];
    float *out[MAXE];
    int len[MAXE], first[MAXE];
    int n, nchunk;
};
__global__ void __launch_bounds__(256) k_sum_parts(const SumArgs A)
{
    const int e = table_entry(A.first, A.n);
    const int i = ((int)blockIdx.x - A.first[e]) * 256 + (int)threadIdx.x;
    const int n = A.len[e];
    if (i >= n) return;
    const float *p = A.part[e] + i;
    float s = 0.f;
#pragma unroll 16
    for (int c = 0; c < A.nchunk; ++c) s += p[(size_t)c * n];
    A.out[e][i] = s;
}

// w'[tap][ci][co] = w[8 - tap][co][ci]: the data gradient is the forward
// convolution of dy with the flipped, transposed kernel
struct FlipArgs {
    const uint16_t *w[MAXL];
    uint16_t *wt[MAXL];
    int cout[MAXL], cin[MAXL], first[MAXL];
    int n;
};
__global__ void __launch_bounds__(256) k_flip_weights(const FlipArgs A)
{
    const int e = table_entry(A.first, A.n);
    const int i = ((int)blockIdx.x - A.first[e]) * 256 + (int)threadIdx.x;
    const int Cout = A.cout[e], Cin = A.cin[e];
    if (i >= 9 * Cout * Cin) return;
    const int tap = i / (Cin * Cout);
    const int r = i - tap * Cin * Cout;
    const int ci = r / Cout, co = r - ci * Cout;
    A.wt[e][i] = A.w[e][((size_t)(8 - tap) * Cout + co) * Cin + ci];
}

// ---------------------------------------------------------------------------
// pooling, upsampling, input and output layers
// ---------------------------------------------------------------------------
// 2x2 average: out (H/2 x W/2) from in (H x W), C channels
__global__ void k_pool2(const uint16_t *__restrict__ in, int cs_in, uint16_t *out, int cs_out,
                        int H, int W, int C)
{
    const int Ho = H / 2, Wo = W / 2;
    const size_t n = (size_t)Ho * Wo * C;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x) {
        const int c = (int)(i % C);
        const size_t p = i / C;
        const int yo = (int)(p / Wo), xo = (int)(p % Wo);
        const size_t b = ((size_t)(2 * yo) * W + 2 * xo) * cs_in + c;
        const float s = (bf2f(in[b]) + bf2f(in[b + cs_in])) +
                        (bf2f(in[b + (size_t)W * cs_in]) + bf2f(in[b + (size_t)W * cs_in + cs_in]));
        out[p * cs_out + c] = f2bf(0.25f * s);
    }
}

// its gradient: din += 0.25 dout (each fine pixel from its coarse pixel)
__global__ void k_pool2_bwd(const uint16_t *__restrict__ dout, int cs_out, uint16_t *din,
                            int cs_in, int H, int W, int C, int accum)
{
    const size_t n = (size_t)H * W * C;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x) {
        const int c = (int)(i % C);
        const size_t p = i / C;
        const int y = (int)(p / W), x = (int)(p % W);
        float v = 0.25f * bf2f(dout[((size_t)(y / 2) * (W / 2) + x / 2) * cs_out + c]);
        uint16_t *o = din + p * cs_in + c;
        if (accum) v += bf2f(*o);
        *o = f2bf(v);
    }
}

// nearest-neighbour 2x upsampling: out (2H x 2W) from in (H x W)
__global__ void k_up2(const uint16_t *__restrict__ in, int cs_in, uint16_t *out, int cs_out,
                      int H, int W, int C)
{
    const int Ho = 2 * H, Wo = 2 * W;
    const size_t n = (size_t)Ho * Wo * C;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x) {
        const int c = (int)(i % C);
        const size_t p = i / C;
        const int y = (int)(p / Wo), x = (int)(p % Wo);
        out[p * cs_out + c] = in[((size_t)(y / 2) * W + x / 2) * cs_in + c];
    }
}

// its gradient: din (H x W) = sum of the 4 fine pixels of dout (2H x 2W)
__global__ void k_up2_bwd(const uint16_t *__restrict__ dout, int cs_out, uint16_t *din,
                          int cs_in, int H, int W, int C)
{
    const size_t n = (size_t)H * W * C;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x) {
        const int c = (int)(i % C);
        const size_t p = i / C;
        const int y = (int)(p / W), x = (int)(p % W);
        const size_t b = ((size_t)(2 * y) * (2 * W) + 2 * x) * cs_out + c;
        const size_t r = (size_t)(2 * W) * cs_out;
        const float s = (bf2f(dout[b]) + bf2f(dout[b + cs_out])) + (bf2f(dout[b + r]) + bf2f(dout[b + r + cs_out]));
        din[p * cs_in + c] = f2bf(s);
    }
}

// input layer: f32 planes [c][H][W] (pitch ld) scaled by scale[c] -> BF16
// NHWC with cs channels (channels >= nc are zero)
__global__ void k_pack_input(const float *__restrict__ planes, int nc, size_t plane, int ld,
                             const float *__restrict__ scale, int H, int W, uint16_t *out, int cs)
{
    const size_t n = (size_t)H * W * cs;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x) {
        const int c = (int)(i % cs);
        const size_t p = i / cs;
        const int y = (int)(p / W), x = (int)(p % W);
        const float v = c < nc ? planes[c * plane + (size_t)y * ld + x] * scale[c] : 0.f;
        out[i] = f2bf(v);
    }
}

struct PlaneSet {
    const void *p[8];
    int ld[8];
};

__global__ void k_block_mean(PlaneSet ps, int nc, int dbl, int f, int H, int W, float *out)
{
    const size_t n = (size_t)nc * H * W;
    const float inv = 1.f / (float)(f * f);
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x) {
        const int X = (int)(i % W);
        const size_t r = i / W;
        const int Y = (int)(r % H), c = (int)(r / H);
        const size_t o = (size_t)f * Y * ps.ld[c] + (size_t)f * X;
        float s = 0.f;
        if ((dbl >> c) & 1) {
            const double *q = (const double *)ps.p[c] + o;
            for (int a = 0; a < f; ++a)
                for (int b = 0; b < f; ++b) s += (float)q[(size_t)a * ps.ld[c] + b];
        } else {
            const float *q = (const float *)ps.p[c] + o;
            for (int a = 0; a < f; ++a)
                for (int b = 0; b < f; ++b) s += q[(size_t)a * ps.ld[c] + b];
        }
        out[i] = s * inv;
    }
}

// bilinear weights of fine node t (0 <= t < f n) between coarse centres
// f T + (f - 1) / 2, clamped at the first and last centre
__device__ __forceinline__ void lin1(int t, int f, int n, int &i0, int &i1, float &w1)
{
    const float u = ((float)t - 0.5f * (float)(f - 1)) / (float)f;
    if (u <= 0.f) { i0 = i1 = 0; w1 = 0.f; return; }
    if (u >= (float)(n - 1)) { i0 = i1 = n - 1; w1 = 0.f; return; }
    i0 = (int)u;
    i1 = i0 + 1;
    w1 = u - (float)i0;
}

template <typename R>
__global__ void k_seed_apply(const float *__restrict__ corr, int H, int W, int f, float s,
                             const float *__restrict__ a, const float *__restrict__ b, int ld_ab,
                             size_t pl_ab, R *dst, int ld_d, size_t pl_d, int ny1, int nx1)
{
    const size_t n = (size_t)2 * ny1 * nx1;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x) {
        const int x = (int)(i % nx1);
        const size_t r = i / nx1;
        const int y = (int)(r % ny1), c = (int)(r / ny1);
        const size_t ab = c * pl_ab + (size_t)y * ld_ab + x;
        float v = a ? 2.f * a[ab] - b[ab] : 0.f;
        if (y < f * H && x < f * W) {
            int y0, y1, x0, x1;
            float wy, wx;
            lin1(y, f, H, y0, y1, wy);
            lin1(x, f, W, x0, x1, wx);
            const float *q = corr + (size_t)c * H * W;
            const float top = (1.f - wx) * q[(size_t)y0 * W + x0] + wx * q[(size_t)y0 * W + x1];
            const float bot = (1.f - wx) * q[(size_t)y1 * W + x0] + wx * q[(size_t)y1 * W + x1];
            v += s * ((1.f - wy) * top + wy * bot);
        }
        dst[c * pl_d + (size_t)y * ld_d + x] = (R)v;
    }
}

template <typename R>
__global__ void k_seed_combine(R *epw, R *hist, const R *__restrict__ corr, size_t n, int extrap)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x) {
        const R e = epw[i];
        if (extrap) epw[i] = corr ? R(2) * e - hist[i] + corr[i] : R(2) * e - hist[i];
        hist[i] = e;
    }
}

// output layer (1x1, cin -> cout <= 4) in FP32: o[c][p] = b[c] + sum_k w[c][k] h[p][k]
__global__ void k_head(const uint16_t *__restrict__ h, int cs, int cin, const float *__restrict__ w,
                       const float *__restrict__ b, int cout, size_t npix, float *o)
{
    for (size_t p = blockIdx.x * (size_t)blockDim.x + threadIdx.x; p < npix;
         p += (size_t)gridDim.x * blockDim.x)
        for (int c = 0; c < cout; ++c) {
            float s = b[c];
            for (int k = 0; k < cin; ++k) s += w[c * cin + k] * bf2f(h[p * cs + k]);
            o[c * npix + p] = s;
        }
}

// head backward: dh[p][k] = sum_c w[c][k] do[c][p] (BF16); per-chunk partial
// weight / bias gradients part[chunk][c][k] and part[chunk][c][cin], each one
// thread's sum over the chunk's pixels in order.  The pixels go through LDS in
// tiles, so that serial sum waits for LDS and not for memory (37 us from memory,
// 10.6 us so, 64 chunks of 256 pixels).
constexpr int HEAD_H = 16384, HEAD_D = 4096;   // tile elements of h and do in LDS
__global__ void __launch_bounds__(256)
k_head_bwd(const uint16_t *__restrict__ h, int cs, int cin, const float *__restrict__ w, int cout,
           size_t npix, const float *__restrict__ dout, uint16_t *dh, int nchunk, int tile,
           int vec, float *part)
{
    __shared__ __attribute__((aligned(16))) uint16_t sh[HEAD_H];
    __shared__ float sd[HEAD_D], sw[256];
    const int chunk = blockIdx.x, t = threadIdx.x;
    if (t < cout * cin) sw[t] = w[t];
    const size_t per = (npix + nchunk - 1) / nchunk;
    const size_t p0 = min(npix, chunk * per), p1 = min(npix, p0 + per);
    const int c = t / (cin + 1), k = t % (cin + 1);
    float s = 0.f;
    for (size_t base = p0; base < p1; base += tile) {
        const int np = (int)min((size_t)tile, p1 - base);
        if (vec) {
            const int kc = cin >> 3;
            uint4 *s4 = reinterpret_cast<uint4 *>(sh);
            for (int i = t; i < np * kc; i += 256)
                s4[i] = *reinterpret_cast<const uint4 *>(h + (base + i / kc) * cs + 8 * (i % kc));
        } else {
            for (int i = t; i < np * cin; i += 256) sh[i] = h[(base + i / cin) * cs + i % cin];
        }
        for (int i = t; i < np * cout; i += 256) sd[i] = dout[(i / np) * npix + base + i % np];
        __syncthreads();
        // thread t < cout*(cin+1) owns one (c, k) sum
        if (t < cout * (cin + 1)) {
            const uint16_t *hp = sh + (k < cin ? k : 0);
            const float *dp = sd + c * np;
#pragma unroll 8
            for (int p = 0; p < np; ++p) {
                const float hv = bf2f(hp[p * cin]);
                s += dp[p] * (k < cin ? hv : 1.f);
            }
        }
        auto grad = [&](int p, int kk) -> uint32_t {
            float v = 0.f;
            for (int cc = 0; cc < cout; ++cc) v += sw[cc * cin + kk] * sd[cc * np + p];
            return f2bf(v);
        };
        if (vec) {
            const int kc = cin >> 3;
            for (int i = t; i < np * kc; i += 256) {
                const int p = i / kc, k0 = 8 * (i % kc);
                uint32_t u[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) u[j] = grad(p, k0 + 2 * j) | grad(p, k0 + 2 * j + 1) << 16;
                *reinterpret_cast<uint4 *>(dh + (base + p) * cs + k0) = uint4{u[0], u[1], u[2], u[3]};
            }
        } else {
            for (int i = t; i < np * cin; i += 256)
                dh[(base + i / cin) * cs + i % cin] = (uint16_t)grad(i / cin, i % cin);
        }
        __syncthreads();
    }
    if (t < cout * (cin + 1)) part[(size_t)chunk * cout * (cin + 1) + t] = s;
}

// mean squared error over n values and its gradient 2 (o - t) / n; the loss
// sum goes to per-block partials (fixed-order sum afterwards)
__global__ void k_mse(const float *__restrict__ o, const float *__restrict__ t, size_t n,
                      float *grad, double *partial)
{
    __shared__ double s[256];
    double acc = 0.0;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x) {
        const float d = o[i] - t[i];
        acc += (double)d * d;
        grad[i] = 2.f * d / (float)n;
    }
    s[threadIdx.x] = acc;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if (threadIdx.x < k) s[threadIdx.x] += s[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = s[0];
}

// Adam step on FP32 master weights, refreshing their BF16 copies (if any): all
// vectors of a network in one launch (30 launches of 2.2 us with the gaps
// between them before, one of 5.5 us now)
struct AdamArgs {
    float *w[MAXE];
    const float *g[MAXE];
    float *m[MAXE], *v[MAXE];
    uint16_t *wb[MAXE];
    int len[MAXE], first[MAXE];
    int n;
    float lr, b1, b2, eps, c1, c2;
};
__global__ void __launch_bounds__(256) k_adam(const AdamArgs A)
{
    const int e = table_entry(A.first, A.n);
    const int i = ((int)blockIdx.x - A.first[e]) * 256 + (int)threadIdx.x;
    if (i >= A.len[e]) return;
    const float b1 = A.b1, b2 = A.b2;
    const float gi = A.g[e][i];
    const float mi = b1 * A.m[e][i] + (1.f - b1) * gi;
    const float vi = b2 * A.v[e][i] + (1.f - b2) * gi * gi;
    A.m[e][i] = mi;
    A.v[e][i] = vi;
    const float wv = A.w[e][i] - A.lr * (mi / A.c1) / (sqrtf(vi / A.c2) + A.eps);
    A.w[e][i] = wv;
    if (A.wb[e]) A.wb[e][i] = f2bf(wv);
}

__global__ void k_to_bf16(const float *__restrict__ a, size_t n, uint16_t *b)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x)
        b[i] = f2bf(a[i]);
}

static void add_sum(SumArgs &a, const float *part, int len, float *out)
{
    const int e = a.n++;
    a.part[e] = part;
    a.out[e] = out;
    a.len[e] = len;
    a.first[e] = e ? a.first[e - 1] + (a.len[e - 1] + 255) / 256 : 0;
}

static int launch_sums(const SumArgs &a, hipStream_t st)
{
    const int blocks = a.n ? a.first[a.n - 1] + (a.len[a.n - 1] + 255) / 256 : 0;
    if (!blocks) return QP_OK;
    hipLaunchKernelGGL(k_sum_parts, dim3(blocks), dim3(256), 0, st, a);
    QP_LAUNCH_CHECK();
    return QP_OK;
}

static dim3 g1(size_t n)
{
    size_t b = (n + 255) / 256;
    if (b > 16384) b = 16384;
    return dim3((unsigned)(b ? b : 1));
}

}  // namespace qp

using namespace qp;

#define NET_CHECK(cond, ...) QP_REQUIRE(cond, QP_ERR_ARG, __VA_ARGS__)
#define RC(expr)              \
    do {                      \
        const int rc_ = expr; \
        if (rc_) return rc_;  \
    } while (0)

// what the convolutions ask of the current device
struct NetDevice {
    size_t lds;   // bytes of a workgroup
    int cus;      // compute units
};
static int net_device(NetDevice *d)
{
    // asking takes 0.3 us of a call's 9, so what a device has is asked once
    struct Known {
        std::atomic<int> lds{0}, cus{0};
    };
    static Known known[64];
    int dev = 0;
    QP_HIP(hipGetDevice(&dev));
    Known *k = dev >= 0 && dev < 64 ? &known[dev] : nullptr;
    int lds = k ? k->lds.load(std::memory_order_relaxed) : 0;
    d->cus = k ? k->cus.load(std::memory_order_relaxed) : 0;
    if (!lds) {
        QP_HIP(hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
        if (k) k->lds.store(lds, std::memory_order_relaxed);
    }
    if (!d->cus) {
        QP_HIP(hipDeviceGetAttribute(&d->cus, hipDeviceAttributeMultiprocessorCount, dev));
        if (k) k->cus.store(d->cus, std::memory_order_relaxed);
    }
    d->lds = (size_t)lds;
    return QP_OK;
}

// dev: the current device, if the caller has asked for it already
static int conv3x3(const NetDevice *dev, hipStream_t st, const uint16_t *x, const uint16_t *mask,
                   int H, int W, int cs_in, int cin, const uint16_t *w, const float *bias,
                   uint16_t *out, int cs_out, int cout, int relu, int accum)
{
    NET_CHECK(x && w && out && H > 0 && W > 0, "qp_net_conv3x3: bad argument");
    NET_CHECK(cin % 16 == 0 && cout % 16 == 0 && cout <= 192 && cin <= cs_in &&
                  cout <= cs_out && cs_in % 4 == 0,
              "qp_net_conv3x3: channels cin %d cout %d (multiples of 16, cout <= 192)", cin, cout);
    if (cout <= 0) return QP_OK;
    NetDevice own;
    if (!dev) {
        RC(net_device(&own));
        dev = &own;
    }
    const int gw = (W + 15) / 16;
    // 16-byte loads of the pixels and weights where they are aligned for it
    const bool al = cs_in % 8 == 0 && !(((uintptr_t)x | (uintptr_t)mask | (uintptr_t)w) & 15);
    const int kt = cin / 16;
    const bool have = kt == 1 || kt == 2 || kt == 3 || kt == 4 || kt == 6 || kt == 8 || kt == 12;
    // four pixel groups a block, or fewer where that leaves compute units without
    // one: a block waits for what it brings to LDS
    int tx = gw >= 3 ? 4 : gw, ty = 4 / tx;
    auto blocks = [&](int x, int y) {
        return (size_t)((H + y - 1) / y) * ((gw + x - 1) / x) * (cout / 16);
    };
    while (tx * ty > 1 && 2 * blocks(tx, ty) <= (size_t)dev->cus) {
        if (ty > 1) ty /= 2;
        else tx /= 2;
    }
    const size_t lds = (size_t)((16 * tx + 2) * (ty + 2) + 144) * (cin / 8 + 1) * 16;
    const bool staged = have && al && lds <= dev->lds;
    const bool wide = staged ? mask && conv_wide_masked(dev->cus, (long long)H * gw, cin, cout)
                             : conv_wide(dev->cus, (long long)H * gw, cin, cout);
    if (staged && !wide) {
        const int nbx = (gw + tx - 1) / tx;
        const dim3 grid((unsigned)((size_t)((H + ty - 1) / ty) * nbx), cout / 16);
        auto launch = [&](auto kern) -> int {
            if (lds > 65536)
                QP_HIP(hipFuncSetAttribute((const void *)kern,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            hipLaunchKernelGGL(kern, grid, dim3(256), lds, st, x, mask, H, W, nbx, tx, ty, cs_in, w,
                               bias, out, cs_out, cout, relu, accum);
            return QP_OK;
        };
        int rc = QP_OK;
#define CONV_CASE(KT) \
    case KT: rc = mask ? launch(k_conv3x3<KT, true>) : launch(k_conv3x3<KT, false>); break
        switch (kt) {
            CONV_CASE(1);
            CONV_CASE(2);
            CONV_CASE(3);
            CONV_CASE(4);
            CONV_CASE(6);
            CONV_CASE(8);
            CONV_CASE(12);
        }
#undef CONV_CASE
        RC(rc);
        QP_LAUNCH_CHECK();
        return QP_OK;
    }
    if (wide) {
        hipLaunchKernelGGL(k_conv3x3_wide, dim3((unsigned)(((size_t)H * gw + 3) / 4)), dim3(256), 0,
                           st, x, mask, H, W, gw, cs_in, cin, w, bias, out, cs_out, cout, relu,
                           accum);
        QP_LAUNCH_CHECK();
        return QP_OK;
    }
    const dim3 grid((unsigned)(((size_t)H * gw + 3) / 4), cout / 16);
    if (mask)
        hipLaunchKernelGGL(k_conv3x3_deep<true>, grid, dim3(256), 0, st, x, mask, H, W, gw, cs_in,
                           cin, w, bias, out, cs_out, cout, relu, accum);
    else
        hipLaunchKernelGGL(k_conv3x3_deep<false>, grid, dim3(256), 0, st, x, mask, H, W, gw,
                           cs_in, cin, w, bias, out, cs_out, cout, relu, accum);
    QP_LAUNCH_CHECK();
    return QP_OK;
}

// bias alone: the partial sums take the weights' place in part
static int bias_layer(hipStream_t st, const qp_net_layer &l, int nchunk, float *part)
{
    WgradArgs a{};
    SumArgs sums{};
    a.n = 1;
    a.nchunk = sums.nchunk = nchunk;
    // its blocks are those of the first 16 input channels
    a.l[0] = WgradLayer{l.x, l.dy, l.yout, nullptr, l.db, nullptr, part,
                        l.cs_x, 16, l.cs_y, l.cout, l.H, l.W, WG_ONE};
    hipLaunchKernelGGL(k_wgrad, dim3(l.cout / 16 * 3 * nchunk), dim3(256), 0, st, a);
    QP_LAUNCH_CHECK();
    add_sum(sums, part, l.cout, l.db);
    return launch_sums(sums, st);
}

// partb: the partial sums of the bias of a single layer, if not in part
static int wgrad_layers(const NetDevice &dev, hipStream_t st, const qp_net_layer *layers, int n,
                        int nchunk, float *part, size_t npart, float *partb)
{
    for (int i0 = 0; i0 < n; i0 += MAXL) {
        WgradArgs a{};
        SumArgs sums{}, sumb{};
        a.n = std::min(MAXL, n - i0);
        a.nchunk = sums.nchunk = sumb.nchunk = nchunk;
        size_t used = 0, waves = 0;
        for (int e = 0; e < a.n; ++e) {
            const qp_net_layer &l = layers[i0 + e];
            const int per = (int)(((size_t)l.H * l.W + nchunk - 1) / nchunk);
            const size_t nw = (size_t)9 * l.cout * l.cin, nb = l.db && !partb ? l.cout : 0;
            // a layer whose partial sums find no room: its blocks take all chunks
            const bool parts = per > WG_WHOLE && part && used + (nw + nb) * nchunk <= npart;
            a.l[e] = WgradLayer{l.x, l.dy, l.yout, l.dw, l.db, nullptr, nullptr,
                                l.cs_x, l.cin, l.cs_y, l.cout, l.H, l.W, parts ? WG_FOUR : WG_ALL};
            if (parts) {
                a.l[e].part = part + used;
                a.l[e].partb = partb ? partb : part + used + nw * nchunk;
                used += (nw + nb) * nchunk;
                if (l.db) add_sum(partb ? sumb : sums, a.l[e].partb, l.cout, l.db);
                add_sum(sums, a.l[e].part, (int)nw, l.dw);
            }
            waves += (size_t)(l.cout / 16) * (l.cin / 16) * 3 * (parts ? nchunk : 4);
        }
        int blocks = 0;
        for (int e = 0; e < a.n; ++e) {
            WgradLayer &l = a.l[e];
            const int per = (l.H * l.W + nchunk - 1) / nchunk;
            if (l.mode == WG_FOUR && waves <= (size_t)wgrad_few(per) * dev.cus) l.mode = WG_ONE;
            a.first[e] = blocks;
            blocks += (l.cout / 16) * (l.cin / 16) * 3 *
                      (l.mode == WG_ALL ? 1 : l.mode == WG_FOUR ? (nchunk + 3) / 4 : nchunk);
        }
        hipLaunchKernelGGL(k_wgrad, dim3(blocks), dim3(256), 0, st, a);
        QP_LAUNCH_CHECK();
        RC(launch_sums(sumb, st));
        RC(launch_sums(sums, st));
    }
    return QP_OK;
}

extern "C" {

int qp_net_conv3x3(void *stream_, const uint16_t *x, const uint16_t *mask, int H, int W,
                   int cs_in, int cin, const uint16_t *w, const float *bias, uint16_t *out,
                   int cs_out, int cout, int relu, int accum)
{
    return conv3x3(nullptr, (hipStream_t)stream_, x, mask, H, W, cs_in, cin, w, bias, out, cs_out,
                   cout, relu, accum);
}

int qp_net_wgrad_layers(void *stream_, const qp_net_layer *layers, int n, int nchunk, float *part,
                        size_t npart)
{
    NET_CHECK((layers || !n) && n >= 0 && nchunk > 0, "qp_net_wgrad_layers: bad argument");
    for (int i = 0; i < n; ++i) {
        const qp_net_layer &l = layers[i];
        NET_CHECK(l.x && l.dy && l.yout && l.dw && l.H > 0 && l.W > 0 && l.cin > 0 && l.cout > 0 &&
                      l.cin % 16 == 0 && l.cout % 16 == 0,
                  "qp_net_wgrad_layers: layer %d", i);
    }
    NetDevice dev;
    RC(net_device(&dev));
    return wgrad_layers(dev, (hipStream_t)stream_, layers, n, nchunk, part, npart, nullptr);
}

int qp_net_conv3x3_wgrad(void *stream_, const uint16_t *x, int cs_in, int cin,
                         const uint16_t *dy, const uint16_t *yout, int cs_out, int cout, int H,
                         int W, int nchunk, float *part, float *dw, float *db)
{
    NET_CHECK(x && dy && yout && part && dw && nchunk > 0, "qp_net_conv3x3_wgrad: bad argument");
    NET_CHECK(cin % 16 == 0 && cout % 16 == 0, "qp_net_conv3x3_wgrad: channels");
    qp_net_layer l = {x, dy, yout, dw, db, cs_in, cin, cs_out, cout, H, W};
    NetDevice dev;
    RC(net_device(&dev));
    // the scratch holds the weights' partial sums; the bias's wait in dw, which is
    // written behind them, or, where they do not fit there, take the scratch first
    // (1024^2 16 -> 16, 200 chunks: 168 us; as one block's chunks 9750)
    const size_t per = ((size_t)H * W + nchunk - 1) / nchunk;
    if (db && nchunk > 9 * cin && cin > 0 && cout > 0 && per > WG_WHOLE) {
        RC(bias_layer((hipStream_t)stream_, l, nchunk, part));
        l.db = nullptr;
    }
    return wgrad_layers(dev, (hipStream_t)stream_, &l, 1, nchunk, part,
                        (size_t)nchunk * 9 * cout * cin, l.db ? dw : nullptr);
}

int qp_net_flip_layers(void *stream_, const qp_net_flip *layers, int n)
{
    hipStream_t st = (hipStream_t)stream_;
    NET_CHECK((layers || !n) && n >= 0, "qp_net_flip_layers: bad argument");
    for (int i = 0; i < n; ++i)
        NET_CHECK(layers[i].w && layers[i].wt, "qp_net_flip_weights: null");
    for (int i0 = 0; i0 < n; i0 += MAXL) {
        FlipArgs a{};
        a.n = std::min(MAXL, n - i0);
        int blocks = 0;
        for (int e = 0; e < a.n; ++e) {
            const qp_net_flip &l = layers[i0 + e];
            a.w[e] = l.w;
            a.wt[e] = l.wt;
            a.cout[e] = l.cout;
            a.cin[e] = l.cin;
            a.first[e] = blocks;
            blocks += (9 * l.cout * l.cin + 255) / 256;
        }
        if (!blocks) continue;
        hipLaunchKernelGGL(k_flip_weights, dim3(blocks), dim3(256), 0, st, a);
        QP_LAUNCH_CHECK();
    }
    return QP_OK;
}

int qp_net_flip_weights(void *stream_, const uint16_t *w, int cout, int cin, uint16_t *wt)
{
    const qp_net_flip l = {w, wt, cout, cin};
    return qp_net_flip_layers(stream_, &l, 1);
}

int qp_net_pool2(void *stream_, const uint16_t *in, int cs_in, uint16_t *out, int cs_out, int H,
                 int W, int C)
{
    hipStream_t st = (hipStream_t)stream_;
    hipLaunchKernelGGL(k_pool2, g1((size_t)H * W * C / 4), dim3(256), 0, st, in, cs_in, out,
                       cs_out, H, W, C);
    QP_LAUNCH_CHECK();
    return QP_OK;
}

int qp_net_pool2_bwd(void *stream_, const uint16_t *dout, int cs_out, uint16_t *din, int cs_in,
                     int H, int W, int C, int accum)
{
    hipStream_t st = (hipStream_t)stream_;
    hipLaunchKernelGGL(k_pool2_bwd, g1((size_t)H * W * C), dim3(256), 0, st, dout, cs_out, din,
                       cs_in, H, W, C, accum);
    QP_LAUNCH_CHECK();
    return QP_OK;
}

int qp_net_up2(void *stream_, const uint16_t *in, int cs_in, uint16_t *out, int cs_out, int H,
               int W, int C)
{
    hipStream_t st = (hipStream_t)stream_;
    hipLaunchKernelGGL(k_up2, g1((size_t)4 * H * W * C), dim3(256), 0, st, in, cs_in, out, cs_out,
                       H, W, C);
    QP_LAUNCH_CHECK();
    return QP_OK;
}

int qp_net_up2_bwd(void *stream_, const uint16_t *dout, int cs_out, uint16_t *din, int cs_in,
                   int H, int W, int C)
{
    hipStream_t st = (hipStream_t)stream_;
    hipLaunchKernelGGL(k_up2_bwd, g1((size_t)H * W * C), dim3(256), 0, st, dout, cs_out, din,
                       cs_in, H, W, C);
    QP_LAUNCH_CHECK();
    return QP_OK;
}

int qp_net_pack_input(void *stream_, const float *planes, int nc, size_t plane, int ld,
                      const float *scale, int H, int W, uint16_t *out, int cs)
{
    hipStream_t st = (hipStream_t)stream_;
    hipLaunchKernelGGL(k_pack_input, g1((size_t)H * W * cs), dim3(256), 0, st, planes, nc, plane,
                       ld, scale, H, W, out, cs);
    QP_LAUNCH_CHECK();
    return QP_OK;
}

int qp_net_block_mean(void *stream_, int nc, const void *const *planes, const int *ld, int dbl,
                      int f, int H, int W, float *out)
{
    hipStream_t st = (hipStream_t)stream_;
    NET_CHECK(nc >= 1 && nc <= 8 && planes && ld && out && f >= 1 && H > 0 && W > 0,
              "qp_net_block_mean: bad argument");
    PlaneSet ps{};
    for (int c = 0; c < nc; ++c) {
        NET_CHECK(planes[c] && ld[c] >= f * W, "qp_net_block_mean: plane %d", c);
        ps.p[c] = planes[c];
        ps.ld[c] = ld[c];
    }
    hipLaunchKernelGGL(k_block_mean, g1((size_t)nc * H * W), dim3(256), 0, st, ps, nc, dbl, f, H,
                       W, out);
    QP_LAUNCH_CHECK();
    return QP_OK;
}

int qp_net_seed_apply(void *stream_, const float *corr, int H, int W, int f, float s,
                      const float *a, const float *b, int ld_ab, size_t pl_ab, void *dst,
                      int dst_double, int ld_d, size_t pl_d, int ny1, int nx1)
{
    hipStream_t st = (hipStream_t)stream_;
    NET_CHECK(corr && dst && H > 0 && W > 0 && f >= 1 && ny1 > 0 && nx1 > 0 && ld_d >= nx1 &&
                  pl_d >= (size_t)ld_d * ny1 && (!a) == (!b) &&
                  (!a || (ld_ab >= nx1 && pl_ab >= (size_t)ld_ab * ny1)),
              "qp_net_seed_apply: bad argument");
    const size_t n = (size_t)2 * ny1 * nx1;
    if (dst_double)
        hipLaunchKernelGGL(k_seed_apply<double>, g1(n), dim3(256), 0, st, corr, H, W, f, s, a, b,
                           ld_ab, pl_ab, (double *)dst, ld_d, pl_d, ny1, nx1);
    else
        hipLaunchKernelGGL(k_seed_apply<float>, g1(n), dim3(256), 0, st, corr, H, W, f, s, a, b,
                           ld_ab, pl_ab, (float *)dst, ld_d, pl_d, ny1, nx1);
    QP_LAUNCH_CHECK();
    return QP_OK;
}

int qp_net_seed_combine(void *stream_, void *epw, void *hist, const void *corr, size_t n,
                        int extrap, int dbl)
{
    hipStream_t st = (hipStream_t)stream_;
    NET_CHECK(epw && hist && n > 0, "qp_net_seed_combine: bad argument");
    if (dbl)
        hipLaunchKernelGGL(k_seed_combine<double>, g1(n), dim3(256), 0, st, (double *)epw,
                           (double *)hist, (const double *)corr, n, extrap);
    else
        hipLaunchKernelGGL(k_seed_combine<float>, g1(n), dim3(256), 0, st, (float *)epw,
                           (float *)hist, (const float *)corr, n, extrap);
    QP_LAUNCH_CHECK();
    return QP_OK;
}

int qp_net_graph_begin(void *stream_)
{
    QP_HIP(hipStreamBeginCapture((hipStream_t)stream_, hipStreamCaptureModeThreadLocal));
    return QP_OK;
}

int qp_net_graph_end(void *stream_, void **graph_exec)
{
    NET_CHECK(graph_exec, "qp_net_graph_end: null output");
    hipGraph_t g = nullptr;
    QP_HIP(hipStreamEndCapture((hipStream_t)stream_, &g));
    hipGraphExec_t ge = nullptr;
    const hipError_t e = hipGraphInstantiate(&ge, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    QP_HIP(e);
    *graph_exec = (void *)ge;
    return QP_OK;
}

int qp_net_graph_launch(void *graph_exec, void *stream_)
{
    NET_CHECK(graph_exec, "qp_net_graph_launch: null graph");
    QP_HIP(hipGraphLaunch((hipGraphExec_t)graph_exec, (hipStream_t)stream_));
    return QP_OK;
}

int qp_net_graph_destroy(void *graph_exec)
{
    if (graph_exec) QP_HIP(hipGraphExecDestroy((hipGraphExec_t)graph_exec));
    return QP_OK;
}

int qp_net_head(void *stream_, const uint16_t *h, int cs, int cin, const float *w,
                const float *b, int cout, size_t npix, float *o)
{
    hipStream_t st = (hipStream_t)stream_;
    hipLaunchKernelGGL(k_head, g1(npix), dim3(256), 0, st, h, cs, cin, w, b, cout, npix, o);
    QP_LAUNCH_CHECK();
    return QP_OK;
}

int qp_net_head_bwd(void *stream_, const uint16_t *h, int cs, int cin, const float *w, int cout,
                    size_t npix, const float *dout, uint16_t *dh, int nchunk, float *part,
                    float *dwb)
{
    hipStream_t st = (hipStream_t)stream_;
    NET_CHECK(cout * (cin + 1) <= 256, "qp_net_head_bwd: head too large");
    // 16 bytes at a time where the pixels are aligned for it
    const int vec = cin % 8 == 0 && cs % 8 == 0 && !(((uintptr_t)h | (uintptr_t)dh) & 15);
    const int tile = std::min(256, std::min(HEAD_H / std::max(cin, 1), HEAD_D / std::max(cout, 1)));
    hipLaunchKernelGGL(k_head_bwd, dim3(nchunk), dim3(256), 0, st, h, cs, cin, w, cout, npix,
                       dout, dh, nchunk, tile, vec, part);
    QP_LAUNCH_CHECK();
    SumArgs a{};
    a.nchunk = nchunk;
    add_sum(a, part, cout * (cin + 1), dwb);
    return launch_sums(a, st);
}

int qp_net_mse(void *stream_, const float *o, const float *t, size_t n, float *grad,
               double *partial, int nblk)
{
    hipStream_t st = (hipStream_t)stream_;
    hipLaunchKernelGGL(k_mse, dim3(nblk), dim3(256), 0, st, o, t, n, grad, partial);
    QP_LAUNCH_CHECK();
    return QP_OK;
}

int qp_net_adam_params(void *stream_, const qp_net_param *params, int n, float lr, float b1,
                       float b2, float eps, int step)
{
    hipStream_t st = (hipStream_t)stream_;
    NET_CHECK((params || !n) && n >= 0, "qp_net_adam_params: bad argument");
    AdamArgs a{};
    a.lr = lr;
    a.b1 = b1;
    a.b2 = b2;
    a.eps = eps;
    a.c1 = 1.f - powf(b1, (float)step);
    a.c2 = 1.f - powf(b2, (float)step);
    int blocks = 0;
    auto flush = [&]() -> int {
        if (blocks) {
            hipLaunchKernelGGL(k_adam, dim3(blocks), dim3(256), 0, st, a);
            QP_LAUNCH_CHECK();
        }
        a.n = blocks = 0;
        return QP_OK;
    };
    for (int i = 0; i < n; ++i) {
        const qp_net_param &p = params[i];
        // a vector longer than an entry can hold goes in pieces
        for (size_t o = 0; o < p.n; o += (size_t)1 << 28) {
            const int len = (int)std::min(p.n - o, (size_t)1 << 28);
            if (a.n == MAXE || blocks > (1 << 20)) RC(flush());
            const int e = a.n++;
            a.w[e] = p.w + o;
            a.g[e] = p.g + o;
            a.m[e] = p.m + o;
            a.v[e] = p.v + o;
            a.wb[e] = p.wb ? p.wb + o : nullptr;
            a.len[e] = len;
            a.first[e] = blocks;
            blocks += (len + 255) / 256;
        }
    }
    return flush();
}

int qp_net_adam(void *stream_, float *wm, const float *g, float *m, float *v, size_t n, float lr,
                float b1, float b2, float eps, int step, uint16_t *wb)
{
    const qp_net_param p = {wm, g, m, v, wb, n};
    return qp_net_adam_params(stream_, &p, 1, lr, b1, b2, eps, step);
}

int qp_net_to_bf16(void *stream_, const float *a, size_t n, uint16_t *b)
{
    hipStream_t st = (hipStream_t)stream_;
    hipLaunchKernelGGL(k_to_bf16, g1(n), dim3(256), 0, st, a, n, b);
    QP_LAUNCH_CHECK();
    return QP_OK;
}

// The U-Net's passes: the launches in order, from one call (22 of a forward and
// 25 of a backward pass took 10 us each from Python, more than most of their
// kernels take).  Level l is the grid coarsened 2^l times; cat[l] holds what the
// decoder convolves there: c[l + 1] channels from below and c[l] from the encoder.
int qp_net_unet_forward(void *st, const qp_net_unet *u, const float *planes, size_t plane, int ld)
{
    NET_CHECK(u && planes, "qp_net_unet_forward: null");
    const qp_net_conv *e = u->enc, *d = u->dec;
    const qp_net_maps &a = u->a;
    const int *c = u->c;
    NetDevice dev;
    RC(net_device(&dev));
    auto conv = [&](const uint16_t *x, int l, int cs, const qp_net_conv &v, uint16_t *out,
                    int cs_out) {
        return conv3x3(&dev, (hipStream_t)st, x, nullptr, u->H >> l, u->W >> l, cs, v.cin, v.w, v.b,
                       out, cs_out, v.cout, 1, 0);
    };
    RC(qp_net_pack_input(st, planes, u->nin, plane, ld, u->in_scale, u->H, u->W, a.x0, 16));
    const uint16_t *in = a.x0;
    int cs = 16;
    for (int l = 0; l < 3; ++l) {
        RC(conv(in, l, cs, e[2 * l], a.ea[l], c[l]));
        RC(conv(a.ea[l], l, c[l], e[2 * l + 1], a.cat[l] + c[l + 1], c[l + 1] + c[l]));
        RC(qp_net_pool2(st, a.cat[l] + c[l + 1], c[l + 1] + c[l], a.pool[l], c[l], u->H >> l,
                        u->W >> l, c[l]));
        in = a.pool[l];
        cs = c[l];
    }
    RC(conv(in, 3, cs, e[6], a.ba, c[3]));
    RC(conv(a.ba, 3, c[3], e[7], a.bb, c[3]));
    in = a.bb;
    for (int l = 2; l >= 0; --l) {
        const qp_net_conv *v = d + 2 * (2 - l);
        RC(qp_net_up2(st, in, c[l + 1], a.cat[l], c[l + 1] + c[l], u->H >> (l + 1),
                      u->W >> (l + 1), c[l + 1]));
        RC(conv(a.cat[l], l, c[l + 1] + c[l], v[0], a.da[l], c[l]));
        RC(conv(a.da[l], l, c[l], v[1], a.db[l], c[l]));
        in = a.db[l];
    }
    return qp_net_head(st, a.db[0], c[0], c[0], u->hw, u->hb, u->nout, (size_t)u->H * u->W, u->out);
}

int qp_net_unet_backward(void *st, const qp_net_unet *u, const float *target)
{
    NET_CHECK(u && target, "qp_net_unet_backward: null");
    const qp_net_conv *e = u->enc, *d = u->dec;
    const qp_net_maps &a = u->a, &g = u->g;
    const int *c = u->c;
    const size_t npix = (size_t)u->H * u->W;
    NetDevice dev;
    RC(net_device(&dev));
    RC(qp_net_mse(st, u->out, target, u->nout * npix, u->gout, u->mse_part, u->nmse));
    RC(qp_net_head_bwd(st, a.db[0], c[0], c[0], u->hw, u->nout, npix, u->gout, g.db[0], u->nhead,
                       u->part, u->ghwb));
    qp_net_flip fl[14];
    for (int i = 0; i < 14; ++i) {
        const qp_net_conv &v = i < 8 ? e[i] : d[i - 8];
        fl[i] = qp_net_flip{v.w, v.wt, v.cout, v.cin};
    }
    RC(qp_net_flip_layers(st, fl + 1, 13));   // the input's gradient is not wanted
    // A convolution's data gradient into gx (if given) from gy, the gradient of its
    // ReLU output y.  Its weight gradient waits for nothing but gy, and all gy are
    // still as their layers left them at the end: one launch for all.
    qp_net_layer wg[14];
    int nwg = 0;
    auto conv = [&](const uint16_t *x, int l, int cs, const qp_net_conv &v, const uint16_t *y,
                    const uint16_t *gy, int cs_y, uint16_t *gx) -> int {
        wg[nwg++] = qp_net_layer{x, gy, y, v.gw, v.gb, cs, v.cin, cs_y, v.cout, u->H >> l, u->W >> l};
        if (!gx) return QP_OK;
        return conv3x3(&dev, (hipStream_t)st, gy, y, u->H >> l, u->W >> l, cs_y, v.cout, v.wt,
                       nullptr, gx, cs, v.cin, 0, 0);
    };
    for (int l = 0; l < 3; ++l) {
        const qp_net_conv *v = d + 2 * (2 - l);
        RC(conv(a.da[l], l, c[l], v[1], a.db[l], g.db[l], c[l], g.da[l]));
        RC(conv(a.cat[l], l, c[l + 1] + c[l], v[0], a.da[l], g.da[l], c[l], g.cat[l]));
        RC(qp_net_up2_bwd(st, g.cat[l], c[l + 1] + c[l], l < 2 ? g.db[l + 1] : g.bb, c[l + 1],
                          u->H >> (l + 1), u->W >> (l + 1), c[l + 1]));
    }
    RC(conv(a.ba, 3, c[3], e[7], a.bb, g.bb, c[3], g.ba));
    RC(conv(a.pool[2], 3, c[2], e[6], a.ba, g.ba, c[3], g.pool[2]));
    for (int l = 2; l >= 0; --l) {
        // the encoder's part of cat[l]: its gradient is the skip's and the pool's
        const int off = c[l + 1], cs = c[l + 1] + c[l];
        RC(qp_net_pool2_bwd(st, g.pool[l], c[l], g.cat[l] + off, cs, u->H >> l, u->W >> l, c[l], 1));
        RC(conv(a.ea[l], l, c[l], e[2 * l + 1], a.cat[l] + off, g.cat[l] + off, cs, g.ea[l]));
        RC(conv(l ? a.pool[l - 1] : a.x0, l, l ? c[l - 1] : 16, e[2 * l], a.ea[l], g.ea[l], c[l],
                l ? g.pool[l - 1] : nullptr));
    }
    return qp_net_wgrad_layers(st, wg, nwg, u->nchunk, u->part, u->npart);
}

}  // extern "C"
