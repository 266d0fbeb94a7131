// k_metropolis.hip -- one checkerboard Metropolis sub-sweep (mu, parity).
//
// Replaces System::update / updateLink (GLAC/system.cpp:321-361): GLAC walks
// the links sequentially; here every link U_mu(x) with x of the given parity
// is updated at once.  Its staple only involves U_mu at the other parity and
// U_nu, nu != mu, none of which change during the sub-sweep, so the links are
// independent and are updated in place.
//
// Per link: the staple A (WilsonGaugeAction::computeStaple,
// GLAC/actions/wilsongaugeaction.cpp:29-53), then n_hit proposals U' = X U
// with X from GLAC's RST construction (GLAC/math/matrices/
// su3matrixgenerator.h:170-321): three SU(2) matrices x0 1 + i x.sigma in
// blocks (0,1), (0,2), (1,2), x0 = sign(r0) sqrt(1 - eps^2),
// x = eps r / |r|, r ~ U(-1/2, 1/2)^4, product R S T or its inverse by a coin.
// dS = -(beta/3) Re tr[(U' - U) A] (wilsongaugeaction.cpp:9, 24-27) is
// evaluated as -(beta/3) (Re tr(U' A) - Re tr(U A)), with Re tr(U A) carried
// from the last accepted hit; accept iff exp(-dS) > u (GLAC/system.cpp:347).
// After the hits the link is optionally reunitarised in FP64, keeping the
// sign of det U (three stored rows may hold GLAC's det = -1 links).  Uniforms
// come from the link's own counter-based stream (rng.hpp): per hit, GLAC's 13
// centred ones for the proposal as 16-bit halves of seven outputs, then one
// 32-bit open one for the test.
#include "kernels.hpp"
#include "proposal.hpp"

namespace glacx {

// The link after its hits, reunitarised in FP64.
template <class T, int R> __device__ __forceinline__ M3<T> reunitarized(const M3<T> &u)
{
    M3<double> d = convert<double>(u);
    if constexpr (R == 2)
        reunitarize<2, true>(d);  // the store keeps rows 0 and 1 only
    else
        reunitarize_keep_det_sign<sizeof(T) == 4>(d);  // det U = +1 or -1 kept
    return convert<T>(d);
}

// What bounds it: FP32 the vector ALU, which is busy all the time (32^4: 5377
// instructions in each of eight wavefronts per SIMD, 72 us at 2.4 GHz; measured
// 70 to 72); FP64 the same unit with two wavefronts.  Wavefronts in flight: with WAVES = 3 per SIMD a block's loads
// fall into the hits of the two others, with four all blocks of a round load
// together and then compute together, and a last block stays alone more often;
// once there are many rounds the blocks are out of step by themselves, and the
// fourth pays.  Microseconds per sub-sweep by blocks per CU, three | four (four
// with compressed links take 116 registers, which they get with no bound on
// WAVES; bounded they are scheduled into 104 and 2 % slower):
//     blocks per CU    4.5   5.1     6     8    10    12    16    20    40    81
//     compressed FP32 48.1  54.2  55.9  68.9  82.6   102   140   177   350   707
//                     51.0  56.1  59.6  72.3  86.3   104   141   175   343   692
//     FP32            56.3  62.5  66.9  85.4   110   134   183   227   445   894
//                     58.8  65.0  68.8  86.0   109   133   180   224   444   880
template <class T, int R, int WAVES>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(1, WAVES))) void metropolis_kernel(
    typename vec2<T>::type *__restrict__ f, Geom g, int mu, int parity, MetroParams prm,
    unsigned long long *__restrict__ count)
{
    const int h = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
    int n = 0;
    if (h < g.vh) {
        const int idx = parity_index(g, parity, h);
        const Site x = site_of(g, idx);
        const M3<T> a = staple<T, R>(f, g, x, mu);
        M3<T> u = load_link<T, R>(f, g, mu, idx);
        Stream rs(prm.seed, (uint32_t)lex_of(g, x), (uint32_t)mu, STREAM_METROPOLIS, prm.sweep);
        const T eps = T(prm.eps);
        const T x0abs = sqrt(T(1) - eps * eps);
        const double bf = prm.beta / 3.0;
        T tra = retrace_mul(u, a);
        int accepted = 0;
#pragma unroll 1
        for (int hit = 0; hit < prm.n_hit; hit++) {
            const M3<T> v = propose_link<T, R>(rst_proposal<T>(rs, x0abs, eps), u);
            const T trv = retrace_mul(v, a);
            const T ds = T(-bf) * (trv - tra);
            if (accept_prob(ds) > rs.open()) {
                u = v;
                tra = trv;
                accepted++;
            }
        }
        if (prm.reunit) u = reunitarized<T, R>(u);
        store_link<T, R>(f, g, mu, idx, u);
        n = accepted;
    }
    add_count(count, blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6), n);
}

// ---- small lattices: one sub-sweep's links do not fill the chip -----------------
// A wavefront of the kernel above is alone on its SIMD there, and its time is
// the chain staple, then n_hit x (proposal, product, test).  Only the products
// and tests are a chain by nature: the staple's planes are independent, and the
// proposals depend on nothing but the link's stream.  So the links of one
// wavefront get a block of STAPLERS + PROPOSERS wavefronts: the proposers form the
// proposals of up to kRoundHits hits (each advancing the stream to its own), the
// others the staple's terms of one plane each (or one wavefront the whole
// staple), all meet in LDS, and wavefront 0 runs the chain.  Every sum and
// product is formed as above, so the results are the same.
//
// FP32 passes the proposed matrices X through LDS (two rows with two stored
// rows); FP64, to keep two blocks per CU, the SU(2) factors' twelve reals and the
// coins as a bit mask per hit.
//
// What bounds it: the chain, and a launch.  Microseconds per sub-sweep (with 2 of
// event timing) by 64-link groups, the kernel above first, then 3 + 5, 1 + 2 and
// 1 + 1 wavefronts (FP64 3 + 3 in place of 3 + 5):
//     groups      compressed FP32           FP32                     FP64
//         64   16.5 11.1 12.7 13.4   17.2 12.7 13.3 14.1   22.3 17.8 16.6 18.8
//        256   16.6 11.3 12.9 13.6   17.4 13.0 13.5 14.4   23.9 18.2 17.5 19.1
//        512   16.8 13.7 13.6 13.9   18.1 15.4 14.5 14.7   24.6 30.8 20.0 20.0
//        768   17.1 17.9 15.0 14.3   18.7 23.2 16.3 15.2   26.9 42.7 35.3 34.9
//       1024   17.0 20.0 17.2 17.2   19.6 25.3 25.5 27.2   29.9 53.8 37.5 36.6
// Each variant is ahead while its blocks find room side by side: one block of
// eight wavefronts per CU, three of two, in FP64 two of three (by their LDS).
constexpr int kRoundHits = 10;  // GLAC's usual number of hits; more go in rounds

template <class T, int R, int STAPLERS> struct SmallLds {
    static constexpr int kReals = sizeof(T) == 8 ? 12 : 6 * R;
    T x[kRoundHits][kReals][64];
    uint32_t test[kRoundHits][64];  // the test's stream output
    unsigned long long coin[kRoundHits];
    T mat[STAPLERS > 1 ? 4 : 1][18][STAPLERS > 1 ? 64 : 1];
};

template <class T> __device__ __forceinline__ void put18(T (&s)[18][64], int lane, const M3<T> &m)
{
#pragma unroll
    for (int e = 0; e < 9; e++) {
        s[2 * e][lane] = m.e[e / 3][e % 3].r;
        s[2 * e + 1][lane] = m.e[e / 3][e % 3].i;
    }
}
template <class T> __device__ __forceinline__ M3<T> get18(const T (&s)[18][64], int lane)
{
    M3<T> m;
#pragma unroll
    for (int e = 0; e < 9; e++) m.e[e / 3][e % 3] = {s[2 * e][lane], s[2 * e + 1][lane]};
    return m;
}

// The two terms of plane (mu, nu) of the staple at x, in the factors whose sums
// staple() adds: with two stored rows the terms themselves; with three the
// left factor of each term's last product.
template <class T, int R> struct StapleTerm {
    M3<T> up, low;
};
template <class T, int R>
__device__ __forceinline__ StapleTerm<T, R> staple_term(const typename vec2<T>::type *__restrict__ f, const Geom &g,
                                                        const Site &x, int mu, int nu)
{
    const Site xpm = site_step(g, x, mu, +1);
    const DirView<T> vmu = dir_view<T>(f, g, mu), vnu = dir_view<T>(f, g, nu);
    const int ipn = site_step(g, x, nu, +1).idx, imn = site_step(g, x, nu, -1).idx;
    const int ipmmn = site_step(g, xpm, nu, -1).idx;
    StapleTerm<T, R> t;
    if constexpr (R == 2) {
        M3<T> p;
        mm<false, true, false, 2>(p, load_rows01<T, R>(vnu, xpm.idx), load_link<T, R>(vmu, ipn));
        mm<false, true, false, 2>(t.up, p, load_link<T, R>(vnu, x.idx));
        rebuild_third_row(t.up);
        mm<true, true, false, 2>(p, load_link<T, R>(vnu, ipmmn), load_link<T, R>(vmu, imn));
        mm<false, false, false, 2>(t.low, p, load_link<T, R>(vnu, imn));
        rebuild_third_row(t.low);
    } else {
        t.up = mul_ad(load_link<T, R>(vnu, xpm.idx), load_link<T, R>(vmu, ipn));
        form(t.up);
        t.low = mul_dd(load_link<T, R>(vnu, ipmmn), load_link<T, R>(vmu, imn));
        form(t.low);
    }
    return t;
}
// a += the two terms, as staple() adds them
template <class T, int R>
__device__ __forceinline__ void add_term(M3<T> &a, const StapleTerm<T, R> &t,
                                         const typename vec2<T>::type *__restrict__ f, const Geom &g, const Site &x,
                                         int nu)
{
    if constexpr (R == 2) {
        add_to(a, t.up);
        add_to(a, t.low);
    } else {
        const DirView<T> vnu = dir_view<T>(f, g, nu);
        mm<false, true, true>(a, t.up, load_link<T, R>(vnu, x.idx));
        form(a);
        mm<false, false, true>(a, t.low, load_link<T, R>(vnu, site_step(g, x, nu, -1).idx));
        form(a);
    }
}

template <class T, int R, int STAPLERS, int PROPOSERS>
__global__ __launch_bounds__(64 * (STAPLERS + PROPOSERS), STAPLERS > 1 ? 4 : 2) void metropolis_small_kernel(
    typename vec2<T>::type *__restrict__ f, Geom g, int mu, int parity, MetroParams prm,
    unsigned long long *__restrict__ count)
{
    static_assert(STAPLERS == 1 || (STAPLERS == 3 && sizeof(T) == 4), "one wavefront for the staple or one per plane");
    __shared__ SmallLds<T, R, STAPLERS> lds;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h_raw = xcd_block(blockIdx.x, gridDim.x) * 64 + lane;
    const bool valid = h_raw < g.vh;
    const int idx = parity_index(g, parity, valid ? h_raw : g.vh - 1);  // idle lanes mirror a real link, store nothing
    const Site x = site_of(g, idx);
    // Every role passes the same barriers: in each round of hits one when its
    // proposals (and in the first round the staple's terms) are in LDS, and
    // between rounds one when the last round's are used up.
    if (wave >= STAPLERS) {
        const T eps = T(prm.eps);
        const T x0abs = sqrt(T(1) - eps * eps);
        Stream rs(prm.seed, (uint32_t)lex_of(g, x), (uint32_t)mu, STREAM_METROPOLIS, prm.sweep);
        int at = 0;  // the stream stands before hit `at`
#pragma unroll 1
        for (int h0 = 0; h0 < prm.n_hit; h0 += kRoundHits) {
            if (h0 > 0) __syncthreads();
            // this wavefront's share of the round's hits, in order
            const int nh = min(kRoundHits, prm.n_hit - h0), j = wave - STAPLERS;
            const int first = nh * j / PROPOSERS, end = nh * (j + 1) / PROPOSERS;
#pragma unroll 1
            for (int h = first; h < end; h++) {
#pragma unroll 1
                for (; at < h0 + h; at++)
#pragma unroll
                    for (int k = 0; k < 8; k++) rs.next();
                T q[14];
#pragma unroll
                for (int k = 0; k < 7; k++) rs.centered_pair<T>(q[2 * k], q[2 * k + 1]);
                cpx<T> ab[6];
                su2_near_unity(q[0], q[1], q[2], q[3], x0abs, eps, ab[0], ab[1]);
                su2_near_unity(q[4], q[5], q[6], q[7], x0abs, eps, ab[2], ab[3]);
                su2_near_unity(q[8], q[9], q[10], q[11], x0abs, eps, ab[4], ab[5]);
                lds.test[h][lane] = rs.next();
                at++;
                if constexpr (sizeof(T) == 8) {
#pragma unroll
                    for (int k = 0; k < 6; k++) {
                        lds.x[h][2 * k][lane] = ab[k].r;
                        lds.x[h][2 * k + 1][lane] = ab[k].i;
                    }
                    const unsigned long long coin = __ballot(q[12] < T(0));
                    if (lane == 0) lds.coin[h] = coin;
                } else {
                    M3<T> xm = rst_product(ab[0], ab[1], ab[2], ab[3], ab[4], ab[5]);
                    xm = q[12] < T(0) ? dagger(xm) : xm;
#pragma unroll
                    for (int k = 0; k < 3 * R; k++) {
                        lds.x[h][2 * k][lane] = xm.e[k / 3][k % 3].r;
                        lds.x[h][2 * k + 1][lane] = xm.e[k / 3][k % 3].i;
                    }
                }
            }
            __syncthreads();
        }
        return;
    }
    M3<T> a = zero3<T>();
    if constexpr (STAPLERS > 1) {
        const int nu = (mu + 1 + wave) & 3;
        const StapleTerm<T, R> t = staple_term<T, R>(f, g, x, mu, nu);
        if (wave > 0) {
            put18(lds.mat[2 * (wave - 1)], lane, t.up);
            put18(lds.mat[2 * (wave - 1) + 1], lane, t.low);
            __syncthreads();
            for (int h0 = kRoundHits; h0 < prm.n_hit; h0 += kRoundHits) {
                __syncthreads();
                __syncthreads();
            }
            return;
        }
        add_term<T, R>(a, t, f, g, x, nu);
    } else {
        a = staple<T, R>(f, g, x, mu);
    }
    M3<T> u = load_link<T, R>(f, g, mu, idx);
    const double bf = prm.beta / 3.0;
    T tra = T(0);
    int accepted = 0;
#pragma unroll 1
    for (int h0 = 0; h0 < prm.n_hit; h0 += kRoundHits) {
        if (h0 > 0) __syncthreads();
        __syncthreads();
        if (h0 == 0) {
            if constexpr (STAPLERS > 1) {
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    const StapleTerm<T, R> t = {get18(lds.mat[2 * k], lane), get18(lds.mat[2 * k + 1], lane)};
                    add_term<T, R>(a, t, f, g, x, (mu + 2 + k) & 3);
                }
            }
            tra = retrace_mul(u, a);
        }
        const int nh = min(kRoundHits, prm.n_hit - h0);
#pragma unroll 1
        for (int h = 0; h < nh; h++) {
            M3<T> xm;
            if constexpr (sizeof(T) == 8) {
                cpx<T> ab[6];
#pragma unroll
                for (int k = 0; k < 6; k++) ab[k] = {lds.x[h][2 * k][lane], lds.x[h][2 * k + 1][lane]};
                xm = rst_product(ab[0], ab[1], ab[2], ab[3], ab[4], ab[5]);
                xm = (lds.coin[h] >> lane) & 1 ? dagger(xm) : xm;
            } else {
#pragma unroll
                for (int k = 0; k < 3 * R; k++) xm.e[k / 3][k % 3] = {lds.x[h][2 * k][lane], lds.x[h][2 * k + 1][lane]};
            }
            const M3<T> v = propose_link<T, R>(xm, u);
            const T trv = retrace_mul(v, a);
            const T ds = T(-bf) * (trv - tra);
            if (accept_prob(ds) > Stream::open_of(lds.test[h][lane])) {
                u = v;
                tra = trv;
                accepted++;
            }
        }
    }
    if (valid) {
        if (prm.reunit) u = reunitarized<T, R>(u);
        store_link<T, R>(f, g, mu, idx, u);
    }
    add_count(count, blockIdx.x, valid ? accepted : 0);
}

__global__ __launch_bounds__(64) void count_sum_kernel(unsigned long long *__restrict__ slots,
                                                       unsigned long long *__restrict__ counts)
{
    unsigned long long *p = slots + (size_t)blockIdx.x * kCountSlots;
    unsigned long long n = 0;
#pragma unroll
    for (int k = threadIdx.x; k < kCountSlots; k += 64) {
        n += p[k];
        p[k] = 0;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) n += __shfl_down(n, off, 64);
    if (threadIdx.x == 0) counts[blockIdx.x] = n;
}

void launch_count_sum(unsigned long long *slots, unsigned long long *counts, int sweeps, hipStream_t s)
{
    count_sum_kernel<<<sweeps, 64, 0, s>>>(slots, counts);
}

template <class T, int R>
void launch_metropolis(void *f, const Geom &g, int mu, int parity, const MetroParams &p, unsigned long long *count,
                       hipStream_t s)
{
    auto *links = (typename vec2<T>::type *)f;
    const int groups = (g.vh + 63) / 64, blocks = (g.vh + kBlock - 1) / kBlock;
    // the table at metropolis_small_kernel
    if constexpr (sizeof(T) == 4) {
        if (groups <= 256)
            metropolis_small_kernel<T, R, 3, 5><<<groups, 64 * 8, 0, s>>>(links, g, mu, parity, p, count);
        else if (groups <= 768)
            metropolis_small_kernel<T, R, 1, 1><<<groups, 64 * 2, 0, s>>>(links, g, mu, parity, p, count);
        else if (blocks <= (R == 2 ? 3072 : 2048))  // the table at metropolis_kernel
            metropolis_kernel<T, R, 3><<<blocks, kBlock, 0, s>>>(links, g, mu, parity, p, count);
        else
            metropolis_kernel<T, R, R == 2 ? 8 : 4><<<blocks, kBlock, 0, s>>>(links, g, mu, parity, p, count);
    } else {
        if (groups <= 512)
            metropolis_small_kernel<T, R, 1, 2><<<groups, 64 * 3, 0, s>>>(links, g, mu, parity, p, count);
        else
            metropolis_kernel<T, R, 2><<<blocks, kBlock, 0, s>>>(links, g, mu, parity, p, count);
    }
}

template void launch_metropolis<float, 3>(void *, const Geom &, int, int, const MetroParams &, unsigned long long *,
                                       hipStream_t);
template void launch_metropolis<float, 2>(void *, const Geom &, int, int, const MetroParams &, unsigned long long *,
                                       hipStream_t);
template void launch_metropolis<double, 3>(void *, const Geom &, int, int, const MetroParams &, unsigned long long *,
                                        hipStream_t);

} // namespace glacx
