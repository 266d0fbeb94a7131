// proposal.hpp -- GLAC's fixed-eps RST proposal and the accept test, shared by
// the plain and the learned Metropolis kernels.
//
// RST (GLAC/math/matrices/su3matrixgenerator.h:170-321): three SU(2)
// matrices x0 1 + i x.sigma, x0 = sign(r0) sqrt(1 - eps^2), x = eps r / |r|,
// r ~ U(-1/2, 1/2)^4, embedded in blocks (0,1), (0,2), (1,2); X = R S T, or
// its inverse when a 13th uniform is negative (draw order r, s, t, coin as
// GLAC).  Accept iff exp(-dS) > u (GLAC/system.cpp:347).
#pragma once
#include "lattice.hpp"
#include "rng.hpp"

namespace glacx {

// 1/sqrt for the proposal's normalisations: the hardware estimate (about
// 1 ulp) for FP32 links, whose products round at that level anyway; the
// correctly rounded library form for FP64 links.  (HIP's rsqrtf evaluates
// through FP64 to round correctly, about ten instructions per call.)
__device__ __forceinline__ float proposal_rsqrt(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ double proposal_rsqrt(double x) { return rsqrt(x); }

// SU(2) near unity from 4 centred uniforms; returns (a, b) with
// matrix [[a, b], [-conj(b), conj(a)]], a = x0 + i x3, b = x2 + i x1.
template <class T>
__device__ __forceinline__ void su2_near_unity(const T r0, const T r1, const T r2, const T r3, T x0abs, T eps,
                                               cpx<T> &a, cpx<T> &b)
{
    T x0 = r0 < T(0) ? -x0abs : x0abs;
    const T sc = eps * proposal_rsqrt(fma(r1, r1, fma(r2, r2, r3 * r3)));  // eps / |r|
    T x1 = r1 * sc, x2 = r2 * sc, x3 = r3 * sc;
    // |x| = 1 up to rounding (x0^2 = 1 - eps^2).  FP64 renormalises as GLAC
    // does; in FP32 a renormalisation through the 1-ulp estimate would leave
    // |x| - 1 at the same ~1e-7 it finds, so it is skipped.
    if constexpr (sizeof(T) == 8) {
        const T inv = proposal_rsqrt(fma(x0, x0, fma(x1, x1, fma(x2, x2, x3 * x3))));
        x0 *= inv;
        x1 *= inv;
        x2 *= inv;
        x3 *= inv;
    }
    a = {x0, x3};
    b = {x2, x1};
}

// a b - c d with c d rounded first, as a product and a fused multiply-add: the
// compiler may not fuse what product() forms, so only a b is left to fuse.  Written as
// fma(a, b, -(c d)) the sign goes into the multiply, which costs the compressed sweep
// 2 to 4 % (32^4 69.2 | 68.9 us with three wavefronts per SIMD, 74.1 | 72.3 with four;
// 32^3 x 64 143.8 | 141.3; three stored rows 32^3 x 28 75.9 | 73.9), and a product made
// opaque by an empty asm up to 2 % with many hits (32^3 x 52, 23 hits, 198.8 | 195.0).
template <class T> __device__ __forceinline__ T product(T a, T b)
{
#pragma clang fp contract(off)
    return a * b;
}
template <class T> __device__ __forceinline__ T cross(T a, T b, T c, T d) { return a * b - product(c, d); }

// X = R S T with r in block (0,1), s in block (0,2), t in block (1,2), each
// [[a, b], [-conj(b), conj(a)]] there.  Which product of a pair is rounded before
// the other is added is written out, so that a proposal has the same bits in
// every kernel: a chain follows its seed whichever of them a lattice's size picks.
template <class T>
__device__ __forceinline__ M3<T> rst_product(cpx<T> ra, cpx<T> rb, cpx<T> sa, cpx<T> sb, cpx<T> ta, cpx<T> tb)
{
    // R_00 S_01 and R_10 S_01
    const T pr = cross(ra.r, sb.r, ra.i, sb.i), pi = fma(ra.r, sb.i, ra.i * sb.r);
    const T qr = cross(-rb.r, sb.r, rb.i, sb.i), qi = cross(rb.i, sb.r, rb.r, sb.i);
    M3<T> x;
    x.e[0][0] = {cross(ra.r, sa.r, ra.i, sa.i), fma(ra.i, sa.r, ra.r * sa.i)};
    x.e[0][1] = {cross(rb.r, ta.r, rb.i, ta.i) + cross(-tb.r, pr, tb.i, pi),
                 fma(rb.i, ta.r, rb.r * ta.i) + cross(tb.i, pr, tb.r, pi)};
    x.e[0][2] = {cross(rb.r, tb.r, rb.i, tb.i) + fma(pr, ta.r, ta.i * pi),
                 fma(rb.r, tb.i, rb.i * tb.r) + cross(pi, ta.r, ta.i, pr)};
    x.e[1][0] = {cross(-rb.r, sa.r, rb.i, sa.i), cross(rb.i, sa.r, rb.r, sa.i)};
    x.e[1][1] = {fma(ra.r, ta.r, ra.i * ta.i) + cross(-tb.r, qr, tb.i, qi),
                 cross(ra.r, ta.i, ra.i, ta.r) + cross(tb.i, qr, tb.r, qi)};
    x.e[1][2] = {fma(ra.r, tb.r, ra.i * tb.i) + fma(qr, ta.r, ta.i * qi),
                 cross(ra.r, tb.i, ra.i, tb.r) + cross(qi, ta.r, ta.i, qr)};
    x.e[2][0] = {-sb.r, sb.i};
    x.e[2][1] = {cross(sa.i, tb.i, sa.r, tb.r), fma(sa.r, tb.i, sa.i * tb.r)};
    x.e[2][2] = {cross(sa.r, ta.r, sa.i, ta.i), cross(-sa.i, ta.r, sa.r, ta.i)};
    return x;
}

// exp(-dS): FP64 libm exp for FP64 links; the hardware base-2 exponential for
// FP32 links, whose dS already carries FP32 rounding.
__device__ __forceinline__ double accept_prob(double ds) { return exp(-ds); }
__device__ __forceinline__ double accept_prob(float ds) { return (double)__expf(-ds); }

template <class T> __device__ __forceinline__ M3<T> dagger(const M3<T> &m)
{
    M3<T> d;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) d.e[i][j] = {m.e[j][i].r, -m.e[j][i].i};
    return d;
}

// The proposed link U' = X U.  With two stored rows (SU(3) links) only rows 0
// and 1 are multiplied and row 2 is rebuilt as conj(row0 x row1).
template <class T, int R> __device__ __forceinline__ M3<T> propose_link(const M3<T> &xm, const M3<T> &u)
{
    if constexpr (R == 2) {
        M3<T> v;
        mm<false, false, false, 2>(v, xm, u);
        rebuild_third_row(v);
        return v;
    } else {
        return mul(xm, u);
    }
}

// GLAC's 13 uniforms in its order (r0..r3, s0..s3, t0..t3, coin) are the 16-bit
// halves of seven stream outputs, low half first (the 14th half is unused):
// seven 32-bit draws per proposal instead of thirteen.
template <class T> __device__ __forceinline__ M3<T> rst_proposal(Stream &rs, T x0abs, T eps)
{
    T q[14];
#pragma unroll
    for (int k = 0; k < 7; k++) rs.centered_pair<T>(q[2 * k], q[2 * k + 1]);
    cpx<T> ra, rb, sa, sb, ta, tb;
    su2_near_unity(q[0], q[1], q[2], q[3], x0abs, eps, ra, rb);
    su2_near_unity(q[4], q[5], q[6], q[7], x0abs, eps, sa, sb);
    su2_near_unity(q[8], q[9], q[10], q[11], x0abs, eps, ta, tb);
    const M3<T> xm = rst_product(ra, rb, sa, sb, ta, tb);
    return q[12] < T(0) ? dagger(xm) : xm;
}

} // namespace glacx
