// Device side of the sine / cosine transforms, shared by the row transforms
// (qp_fft.hip) and the slice loop's fused spectral kernels (qp_spectral.hip).
// The method and its conventions are described in qp_fft.hip.
#pragma once

#include <type_traits>

#include "qp_common.h"

namespace qp {

// base[i] of a uniform base with a 32-bit byte offset per lane (a plane is far
// below 4 GiB), which the memory instructions add themselves
template <typename T> __device__ __forceinline__ T &at(T *base, unsigned i)
{
    typedef typename std::conditional<std::is_const<T>::value, const char, char>::type C;
    return *reinterpret_cast<T *>(reinterpret_cast<C *>(base) + (unsigned)(i * sizeof(T)));
}

// Every kernel that runs these transforms gives the same bits.  Which product of a
// sum the compiler fuses depends on the kernel around the transform (what becomes
// of an output, and in which block), so the fused ones are written out here, in
// dft8 and in the order of the twiddles' factors; nothing else can be fused.
template <typename R>
__device__ __forceinline__ cplx<R> cmul(cplx<R> a, cplx<R> b)
{
    return {fmadd(a.x, b.x, -(a.y * b.y)), fmadd(a.x, b.y, a.y * b.x)};
}
template <typename R>
__device__ __forceinline__ cplx<R> cadd(cplx<R> a, cplx<R> b) { return {a.x + b.x, a.y + b.y}; }
template <typename R>
__device__ __forceinline__ cplx<R> csub(cplx<R> a, cplx<R> b) { return {a.x - b.x, a.y - b.y}; }
// -i z
template <typename R>
__device__ __forceinline__ cplx<R> cmi(cplx<R> a) { return {a.y, -a.x}; }

// forward DFT of 4 points in place (natural order)
template <typename R>
__device__ __forceinline__ void dft4(cplx<R> &a0, cplx<R> &a1, cplx<R> &a2, cplx<R> &a3)
{
    cplx<R> t0 = cadd(a0, a2), t1 = csub(a0, a2), t2 = cadd(a1, a3), t3 = cmi(csub(a1, a3));
    a0 = cadd(t0, t2);
    a1 = cadd(t1, t3);
    a2 = csub(t0, t2);
    a3 = csub(t1, t3);
}

// forward DFT of 8 points in place (natural order): decimation in frequency,
// X[2m] = DFT4(v[n] + v[n+4]), X[2m+1] = DFT4((v[n] - v[n+4]) w^n), w = e^{-i pi/4}.
// Of the odd outputs' products with 1/sqrt 2 the ones fused are those that the
// row transforms (k_fft_rows) have always fused: in the last pass, which stores
// its outputs one by one (LAST), not those of t3.
template <bool LAST = false, typename R>
__device__ __forceinline__ void dft8(cplx<R> *v)
{
#pragma clang fp contract(off)
    const R h = (R)0.70710678118654752440;
    cplx<R> a0 = cadd(v[0], v[4]), a1 = cadd(v[1], v[5]), a2 = cadd(v[2], v[6]),
            a3 = cadd(v[3], v[7]);
    const cplx<R> c0 = csub(v[0], v[4]), c1 = csub(v[1], v[5]), c2 = cmi(csub(v[2], v[6])),
                  c3 = csub(v[3], v[7]);
    dft4(a0, a1, a2, a3);
    const cplx<R> s1 = {c1.x + c1.y, c1.y - c1.x};                     // c1 e^{-i pi/4} = s1 h
    const cplx<R> p3 = {(c3.y - c3.x) * h, -(c3.x + c3.y) * h};        // c3 e^{-3i pi/4}
    const cplx<R> t0 = cadd(c0, c2), t1 = csub(c0, c2);
    const cplx<R> t2 = {fmadd(s1.x, h, p3.x), fmadd(s1.y, h, p3.y)};
    const cplx<R> d = LAST ? cplx<R>{s1.x * h - p3.x, s1.y * h - p3.y}
                           : cplx<R>{fmadd(s1.x, h, -p3.x), fmadd(s1.y, h, -p3.y)};
    const cplx<R> t3 = cmi(d);
    v[0] = a0; v[2] = a1; v[4] = a2; v[6] = a3;
    v[1] = cadd(t0, t2); v[3] = cadd(t1, t3); v[5] = csub(t0, t2); v[7] = csub(t1, t3);
}

// LDS index of FFT point i: one pad point after every 2^PS points
template <int PS> __device__ __forceinline__ int padk(int i) { return i + (i >> PS); }

// LDS padding by default: one pad point per 16 points in FP32 (a third fewer
// LDS bank conflicts than per 8 at 2048 points), per 8 in FP64
template <typename R> constexpr int pad_shift() { return sizeof(R) == 4 ? 4 : 3; }

template <int L, int PS = 3> struct FftShape {
    static constexpr int M = 1 << L;                // complex points
    static constexpr int N = M / 2;                 // transform length n
    static constexpr int TF = M / 8;                // threads per transform
    static constexpr int BS = TF > 256 ? TF : 256;  // threads per block
    static constexpr int FB = BS / TF;              // transforms per block
    static constexpr int NR8 = L / 3;               // radix-8 passes
    static constexpr int REM = L % 3;               // closing radix-2 (1) / radix-4 (2)
    static constexpr int LDSM = M + (M >> PS) + 1;  // padded LDS points per transform
};

// The twiddles of every pass after the first for thread t: pass p (Ns = 8^p)
// needs W^(r e), e = (t mod Ns) M / (8 Ns), r = 1..7: W^e, W^2e and W^4e come
// from the table W (exp(-2 pi i j / M)), the other four are their products;
// the closing radix-4 pass needs W^j, W^2j (table) and W^3j, the closing
// radix-2 pass W^j
template <typename R, int L> struct Twiddles {
    using S = FftShape<L>;
    cplx<R> w8[S::NR8 > 1 ? 3 * (S::NR8 - 1) : 1];
    cplx<R> wr[S::REM ? 4 : 1];
    __device__ __forceinline__ void load(const cplx<R> *__restrict__ W, int t)
    {
#pragma unroll
        for (int p = 1; p < S::NR8; ++p) {
            const int Ns = 1 << (3 * p);
            const int e = (t & (Ns - 1)) * (S::M / (8 * Ns));
            w8[3 * (p - 1)] = at(W, e);
            w8[3 * (p - 1) + 1] = at(W, 2 * e);
            w8[3 * (p - 1) + 2] = at(W, 4 * e);
        }
        if (S::REM == 2) {
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                wr[2 * s] = at(W, t + s * S::TF);
                wr[2 * s + 1] = at(W, 2 * (t + s * S::TF));
            }
        } else if (S::REM == 1) {
#pragma unroll
            for (int s = 0; s < 4; ++s) wr[s] = at(W, t + s * S::TF);
        }
    }
};

// Position of extension point idx = t + r TF, r = 0..7, in the n + 1 points
template <int L> __device__ __forceinline__ int ext_pos(int idx)
{
    return idx <= FftShape<L>::N ? idx : FftShape<L>::M - idx;
}

// The M-point FFT of one transform by its TF threads: v holds the extension
// points t + r TF; on return z[i] is output point t + i TF (i = 0..3) and zn,
// for t = 0, point N: the outputs that an even or odd extension needs.  buf:
// LDSM points of LDS, all threads of the block take part in its barriers, and
// a barrier is needed before buf is written again.
template <typename R, int L, int PS>
__device__ __forceinline__ void fft_core(cplx<R> (&v)[8], cplx<R> *buf, int t,
                                         const Twiddles<R, L> &tw, cplx<R> (&z)[4], cplx<R> &zn)
{
    using S = FftShape<L, PS>;
    constexpr int M = S::M, TF = S::TF;
    static_assert(S::NR8 > 1 || S::REM != 0, "at least two passes");
    dft8(v);
    // first pass output (Ns = 1): index 8 t + r
#pragma unroll
    for (int r = 0; r < 8; ++r) buf[padk<PS>(8 * t + r)] = v[r];
    // middle radix-8 passes
#pragma unroll
    for (int p = 1; p < S::NR8; ++p) {
        const int Ns = 1 << (3 * p);
        __syncthreads();
        {
            const cplx<R> w1 = tw.w8[3 * (p - 1)], w2 = tw.w8[3 * (p - 1) + 1],
                          w4 = tw.w8[3 * (p - 1) + 2];
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
            // last pass (Ns = M/8): output index t + r M/8
            dft8<true>(v);
#pragma unroll
            for (int i = 0; i < 4; ++i) z[i] = v[i];
            zn = v[4];
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
        // closing radix 4 (Ns = M/4): butterflies t and t + TF
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int j = t + s * TF;
            const cplx<R> w1 = tw.wr[2 * s], w2 = tw.wr[2 * s + 1];
            cplx<R> a0 = buf[padk<PS>(j)];
            cplx<R> a1 = cmul(buf[padk<PS>(j + M / 4)], w1);
            cplx<R> a2 = cmul(buf[padk<PS>(j + M / 2)], w2);
            cplx<R> a3 = cmul(buf[padk<PS>(j + 3 * M / 4)], cmul(w2, w1));
            dft4(a0, a1, a2, a3);
            z[s] = a0;
            z[s + 2] = a1;
            if (s == 0) zn = a2;
        }
    } else {
        // closing radix 2 (Ns = M/2): butterflies t + s TF
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int j = t + s * TF;
            cplx<R> a0 = buf[padk<PS>(j)];
            cplx<R> a1 = cmul(buf[padk<PS>(j + M / 2)], tw.wr[s]);
            z[s] = cadd(a0, a1);
            if (s == 0) zn = csub(a0, a1);
        }
    }
}

// The extension point idx of a row pair's values (a, b) at ext_pos(idx), for
// a sine (type 0) or cosine (1) transform
template <typename R, int L>
__device__ __forceinline__ cplx<R> ext_value(int type, int idx, R a, R b)
{
    constexpr int N = FftShape<L>::N;
    if (type == 0) {
        const int e = ext_pos<L>(idx);
        const bool edge = e == 0 || e == N;
        const R sg = idx > N ? R(-1) : R(1);
        a = edge ? R(0) : sg * a;
        b = edge ? R(0) : sg * b;
    }
    return {a, b};
}

// The two rows' transform values at mode k from the FFT's output point k;
// half: half the transform's scale
template <typename R, int L>
__device__ __forceinline__ cplx<R> row_values(int type, int k, cplx<R> z, R half)
{
    if (type == 1) return {z.x * half, z.y * half};
    if (k == 0 || k == FftShape<L>::N) return {R(0), R(0)};
    return {-z.y * half, z.x * half};
}

}  // namespace qp
