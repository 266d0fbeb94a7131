// k_flow.hip -- one fused stage of Luscher's RK3 Wilson flow.
//
// GLAC's Flow::flowField (GLAC/flow/flow.cpp:43-73) runs each stage as four
// whole-lattice getActionDerivative passes (GLAC/actions/wilsongaugeaction.cpp:
// 55-86), a scale/combine pass, and four matrixExp passes (flow.cpp:95-115),
// each materialising lattice temporaries.  Here a stage is one kernel per
// link: staple -> Omega = U A -> Z = -P_TA(Omega) -> RK3 combination with the
// accumulator -> exp (FP64 Cayley-Hamilton coefficients) -> X U, reading the
// field from `win` and writing `wout` (ping-pong, so every Z of a stage sees
// the same field, as GLAC's separate loops do).
//
//   stage 0:  acc <- Z0                       W1 = exp(eps/4 Z0) W0
//   stage 1:  Y = 8/9 eps Z1 - 17/36 eps acc;  acc <- Y;  W2 = exp(Y) W1
//   stage 2:  Y = 3/4 eps Z2 - acc;                      W3 = exp(Y) W2
//
// The accumulator holds the 8 real parameters of an su(3) element per link
// (16-byte vectors, see acc_store).
//
// FP32 links are reunitarised (FP64 Gram-Schmidt) as the last stage of a
// step stores them.
//
// Launch: 256-thread blocks = 64 sites x 4 directions; wavefront w handles
// mu = w for the block's 64 sites, the h-th to (h+31)-th of each parity (two
// contiguous runs of plane entries, side by side in the lattice).  Even and
// odd sites are neighbours of each other, so a block reads the links around
// one spot of both parity halves, and the four links of a site -- which
// share most staple links -- are processed on the same CU at the same time.
#include "expsu3.hpp"
#include "kernels.hpp"
#include "ldsmat.hpp"

namespace glacx {

// Links a block shares through LDS: wavefront mu loads U_mu(x) (its own
// link) and U_mu(x - mu) for the block's 64 sites; the other three
// wavefronts take them from here for their staples instead of gathering them
// again (U_nu(x) closes every upper staple, U_nu(x - nu) every lower one).
// Per site that is 56 link gathers from memory instead of 76.
// slots 0..3: U_mu(x) for mu = 0..3, slots 4..7: U_mu(x - mu)
template <class T> using FlowLds = LdsMats<T, 8>;

// RK3 accumulator: the 8 real parameters (a0, a1, p0..p5) of an su(3)
// element per link, in 16-byte vectors: two float4 planes per direction in
// FP32 (a0 a1 p0 p1 | p2 p3 p4 p5), four double2 planes in FP64.  Each link's
// wavefront alone touches its entry, once per launch, and nobody reads a link that
// the launch stores.  Stored and loaded as non-temporal (kStreamAcc, kStreamLinks) they
// leave the caches to the links that neighbouring blocks gather; while the Infinity
// Cache's 256 MiB hold what the next stage reads, that throws away what it would
// find there.  So the accumulator is streamed once the two fields and it take
// 256 MiB, the links once the two fields alone exceed that.  Both are also while
// fields and accumulator fit in the eight L2s (32 MiB) or nearly, where a launch
// otherwise ends with writing out what they hold: two fields below 28 MiB in
// FP32; below 16 in FP64, whose gathers find less in a cache that streams.
// Microseconds of a plain stage, with nothing, the accumulator, and both streamed:
//     MiB of two fields, with accumulator    nothing     acc    both
//     compressed  10 x 16^2 x 12    11   15      10.9            10.4
//                 16^3 x 12         18   24      14.0            13.3
//                 16^4              24   32      17.5            17.3
//                 16^2 x 18^2       30   41      22.3            22.9
//                 16^3 x 24         36   48      23.2            24.3
//                 16^2 x 32 x 48   144  192      81.0    84.8    87.7
//                 32^3 x 16        192  256     115.8   114.1   117.5
//                 24^3 x 48        243  324     163.8   145.5   160.1
//                 32^3 x 24        288  384     189.0   183.9   179.6
//                 48^3 x 96       3888 5184      2633    2593    2555
//     FP32        12x10x14x18       17   20      12.9            11.8
//                 16^3 x 12         27   33      16.7            16.2
//                 14x18x22x10       30   37      21.0            21.2
//                 16^2 x 18^2       46   56      26.8            28.8
//                 24^4             182  223      89.6    96.3   109.1
//                 32^3 x 16        288  352     168.1   160.9   162.9
//                 32^4             576  704       344     323     315
//     FP64        8^3 x 16           9   11      11.7            11.5
//                 10 x 12^2 x 10    16   19      12.8            12.8
//                 12^4              23   28      17.3            18.0
//                 16^4              72   88      33.6            37.6
//                 16^3 x 32        144  176      65.9    70.6    75.4
//                 16^3 x 48        216  264     101.7   100.2   109.3
//                 24^3 x 48        729  891     390.2   380.1   370.1
enum StreamBits : unsigned { kStreamAcc = 1, kStreamLinks = 2 };
// The kernels take the bits as a template parameter: tested at run time they cost
// a stage of a small lattice 0.1 to 0.2 us (8^4 compressed 7.93 us without, 8.11 with).
using AccVec = unsigned __attribute__((ext_vector_type(4)));
template <bool STREAM, class V> __device__ __forceinline__ V acc_get(const V *p)
{
    if constexpr (STREAM)
        return __builtin_bit_cast(V, __builtin_nontemporal_load(reinterpret_cast<const AccVec *>(p)));
    else
        return *p;
}
template <bool STREAM, class V> __device__ __forceinline__ void acc_put(V *p, const V &v)
{
    if constexpr (STREAM)
        __builtin_nontemporal_store(__builtin_bit_cast(AccVec, v), reinterpret_cast<AccVec *>(p));
    else
        *p = v;
}
template <bool STREAM>
__device__ __forceinline__ void acc_store(float *acc, const Geom &g, int mu, int idx, const su3alg<float> &z)
{
    float4 *q = reinterpret_cast<float4 *>(acc) + (size_t)mu * 2 * g.v + idx;
    acc_put<STREAM>(q, make_float4(z.a0, z.a1, z.p[0], z.p[1]));
    acc_put<STREAM>(q + g.v, make_float4(z.p[2], z.p[3], z.p[4], z.p[5]));
}
template <bool STREAM>
__device__ __forceinline__ su3alg<float> acc_load(const float *acc, const Geom &g, int mu, int idx)
{
    const float4 *q = reinterpret_cast<const float4 *>(acc) + (size_t)mu * 2 * g.v + idx;
    const float4 u = acc_get<STREAM>(q), v = acc_get<STREAM>(q + g.v);
    su3alg<float> z;
    z.a0 = u.x, z.a1 = u.y, z.p[0] = u.z, z.p[1] = u.w, z.p[2] = v.x, z.p[3] = v.y, z.p[4] = v.z, z.p[5] = v.w;
    return z;
}
template <bool STREAM>
__device__ __forceinline__ void acc_store(double *acc, const Geom &g, int mu, int idx, const su3alg<double> &z)
{
    double2 *q = reinterpret_cast<double2 *>(acc) + (size_t)mu * 4 * g.v + idx;
    acc_put<STREAM>(q, make_double2(z.a0, z.a1));
#pragma unroll
    for (int k = 0; k < 3; k++) acc_put<STREAM>(q + (size_t)(k + 1) * g.v, make_double2(z.p[2 * k], z.p[2 * k + 1]));
}
template <bool STREAM>
__device__ __forceinline__ su3alg<double> acc_load(const double *acc, const Geom &g, int mu, int idx)
{
    const double2 *q = reinterpret_cast<const double2 *>(acc) + (size_t)mu * 4 * g.v + idx;
    su3alg<double> z;
    const double2 u = acc_get<STREAM>(q);
    z.a0 = u.x, z.a1 = u.y;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const double2 v = acc_get<STREAM>(q + (size_t)(k + 1) * g.v);
        z.p[2 * k] = v.x, z.p[2 * k + 1] = v.y;
    }
    return z;
}

// ---- clover observables fused into stage 0 -------------------------------
// Stage 0 of a flow step reads the field the previous step produced, which is
// the field GLAC measures between steps (GLAC/system.cpp:497-503).  Its staple
// terms already hold three of the four clover leaves at x: for wavefront mu
// and term nu, with
//   up  = U_nu(x+mu) U_mu(x+nu)^dag U_nu(x)^dag,
//   low = U_nu(x+mu-nu)^dag U_mu(x-nu)^dag U_nu(x-nu),
// U_mu(x) up is the leaf L1 of plane (mu, nu), U_mu(x) low its leaf L2 and
// also L4^dag of plane (nu, mu) (GLAC's leaves, GLAC/observables/
// mastersamplertopcxyz.cpp:255-328).  The clover C = L1 - L2 + L3 - L4 enters
// the observables only through F = traceless(C - C^dag) (:331-340), which is
// linear in the leaves; with T(M) = traceless(M - M^dag) and T(-M) = T(M^dag),
//   F = T(U_mu(x) (up - low)) + T(L3) + T(U_nu(x) low'),
// low' being wavefront nu's lower term for mu.  So for each of GLAC's planes
// (0,1) (0,2) (0,3) (2,3) (3,1) (1,2) the first-index wavefront adds
// T(U_mu (up - low)), the second-index one T(U_nu low'), and one of the two
// also T(L3), L3 = U_mu(x-mu)^dag U_nu(x-mu-nu)^dag U_mu(x-mu-nu) U_nu(x-nu)
// (two more gathers; both backward links are in LDS).  Every wavefront forms
// one extra product per term, and the L3 leaves are dealt 2, 2, 1, 1.
//
// F of a plane is 8 reals {Im F00, Im F11, F01, F02, F12} in one LDS slot
// per plane.  The three staple terms run as three phases, in a per-wavefront
// order in which the two wavefronts of a plane reach it in different phases: the
// earlier one stores its contribution, the later one holds its own back and adds
// it when all three phases of all are done, so that no wavefront waits for
// another between them (with a barrier after each phase and the sum formed there,
// 32^4 compressed took 398 us for 378, 48^3 x 96 4120 for 3750; the barrier stands
// before the exponential, whose registers are then free of what was held: behind
// it 389).  No atomics, and the sum of the two is formed in a fixed order.  The L3
// leaves go two per phase.  At the end wavefront w < 3 evaluates the pair
// (w, w + 3) = ((0, w+1), (rho, sigma)) per site as the clover kernel does:
//   E += Re tr(F_a F_a) + Re tr(F_b F_b),  q -= Re tr(F_a F_b),
// and the plaquette sum takes Re tr L1 of each plane from its first-index
// wavefront.  The block's sums go to the clover kernel's (chunk, t) slot.

// Slot of GLAC's plane {d1, d2} stored as (d1, d2): 0..2 = (0, nu), 3 = (2,3),
// 4 = (3,1), 5 = (1,2); (mu, nu) is stored as such when mu = 0 or nu = mu % 3 + 1.
__device__ __forceinline__ bool plane_first(int mu, int nu) { return mu == 0 || nu == mu % 3 + 1; }
__device__ __forceinline__ int plane_slot(int d1, int d2) { return d1 == 0 ? d2 - 1 : (d1 == 1 ? 5 : d1 + 1); }
// Phase schedule, entry e = 3 mu + k for wavefront mu in phase k:
//   kPhaseNu:  the term nu (4 bits each): mu 0: 1 2 3, mu 1: 2 0 3, mu 2: 0 3 1, mu 3: 0 1 2
//   kPhaseAdd: the plane's other wavefront stored first (hold, and add at the end)
//   kPhaseL3:  this wavefront also adds the plane's L3 leaf
constexpr unsigned long long kPhaseNu = 0x210130302321ull;
constexpr unsigned kPhaseAdd = 0x936u;  // entries 1 2 4 5 8 11
constexpr unsigned kPhaseL3 = 0x3a3u;   // entries 0 1 5 7 8 9

// SU(3) product from the first two rows of `a` (all that load_rows01 reads):
// the product's first two rows, then its third rebuilt from them.
template <bool DB, class T> __device__ __forceinline__ M3<T> su3_product(const M3<T> &a, const M3<T> &b)
{
    M3<T> p;
    mm<false, DB, false, 2>(p, a, b);
    rebuild_third_row(p);
    return p;
}

template <class T> struct FlowMeasLds {
    T f[6][8][kFlowSites];
};
template <class T> __device__ __forceinline__ FlowMeasLds<T> &flow_meas_lds()
{
    __shared__ FlowMeasLds<T> s;
    return s;
}

// The end of a stage for one link: RK3 combination of the force z with the
// accumulator, exp, product with the link u, and in FP32 the projection.
template <class T, int R, int STAGE, unsigned STREAM>
__device__ __forceinline__ void finish_link(typename vec2<T>::type *__restrict__ wout, T *__restrict__ acc,
                                            const Geom &g, int mu, int idx, const M3<T> &u, const su3alg<T> &z,
                                            const su3alg<T> &cacc, T cz, T ca)
{
    su3alg<T> y;
    if constexpr (STAGE == 0) {
        acc_store<(STREAM & kStreamAcc) != 0>(acc, g, mu, idx, z);
        y.a0 = cz * z.a0;
        y.a1 = cz * z.a1;
#pragma unroll
        for (int k = 0; k < 6; k++) y.p[k] = cz * z.p[k];
    } else {
        y.a0 = cz * z.a0 - ca * cacc.a0;
        y.a1 = cz * z.a1 - ca * cacc.a1;
#pragma unroll
        for (int k = 0; k < 6; k++) y.p[k] = cz * z.p[k] - ca * cacc.p[k];
        if (STAGE == 1) acc_store<(STREAM & kStreamAcc) != 0>(acc, g, mu, idx, y);
    }
    M3<T> w = zero3<T>();
    mm<false, false, false, R>(w, exp_su3(y), u);  // two rows suffice when two are stored
    if constexpr (sizeof(T) == 4 && STAGE == 2) {
        // FP32 links: project back onto the group in FP64 once per flow
        // step, as the last stage stores them.  Without it the rounding of
        // exp(Y) W drifts the links off it (|U U^dag - 1| ~ 1e-4 after 1000
        // steps at 24^3 x 48), and that drift, not the FP32 measurement,
        // dominates the error of E(t) at large t; within a step the two
        // unprojected stores add two roundings (~1e-7), which the
        // projection then removes.  Three stored rows are orthonormalised
        // row by row, which keeps det U (GLAC's det = -1 starts stay
        // det = -1); two stored rows are SU(3) and the third is rebuilt on
        // load.
        M3<double> d = convert<double>(w);
        if constexpr (R == 2)
            reunitarize<2, true>(d);
        else
            orthonormalize_rows<true>(d);
        w = convert<T>(d);
    }
    store_link<T, R, (STREAM & kStreamLinks) != 0>(dir_view<T>(wout, g, mu), idx, w);
}

// Z = -1/2 T(U A), the form force_from_omega evaluates
template <class T> __device__ __forceinline__ su3alg<T> force_from_ta2(const T (&t)[8])
{
    su3alg<T> z;
    z.a0 = T(-0.5) * t[0];
    z.a1 = T(-0.5) * t[1];
#pragma unroll
    for (int k = 0; k < 6; k++) z.p[k] = T(-0.5) * t[2 + k];
    return z;
}

// The end of a measuring stage, by its four wavefronts: wavefront mu < 3 gives F
// of its pair of planes per site, all the plaquette sums; the block's sums go
// to its chunk's slot.
template <class T>
__device__ __forceinline__ void measure_block(const Geom &g, int hb, int mu, T plaq, const T (&fa)[8], const T (&fb)[8],
                                              double *__restrict__ meas)
{
    double s[kMeasAcc] = {(double)plaq, 0.0, 0.0, 0.0};
    if (mu < 3) {
        s[1] = retrace_ta2(fa, fa) + retrace_ta2(fb, fb);
        s[2] = -retrace_ta2(fa, fb);
    }
    block_sum<kMeasAcc>(s);
    if (threadIdx.x == 0) {
        // the block's 32 sites per parity are chunk jc of the run (blk, lt)
        const int h0 = hb * (kFlowSites / 2);
        const int blk = fdiv(h0, g.d_bh);
        const int rem = h0 - blk * g.bh;
        const int lt = fdiv(rem, g.d_run);
        const int jc = (rem - lt * g.run) >> 5;
        const int bt = fdiv(blk, g.d_nzb), zb = blk - bt * g.nzb;
        double *o = meas + kMeasAcc * ((zb * g.cpr + jc) * g.n[3] + (bt << g.lbt) + lt);
#pragma unroll
        for (int i = 0; i < kMeasAcc; i++) o[i] = s[i];
    }
}

// FP64 tuning knob (build time): waves per SIMD the plain stages are compiled for.
#ifndef GLACX_FP64_FLOW_WAVES
#define GLACX_FP64_FLOW_WAVES 2
#endif
// FP64 plain stages of at most kFewBlocks blocks gather a term's links in two pairs and
// all from memory: their wavefronts have at most two SIMD-mates, and what they wait
// for is the first pair, behind which the other loads and the look for near links
// only queue.  Larger launches are bound by requests (see near_slot) and have all four
// in flight.  Microseconds of a stage by blocks, few and many:
//     blocks      1      64     324     480     768     850    1024    1296    1980
//     few        8.3   11.2    17.3    18.9    26.6    33.2    33.6    46.6    66.3
//     many       9.3   11.4    18.6    19.4    27.2    33.2    33.6    45.6    62.7
constexpr int kFewBlocks = 768;

template <class T, int R, int STAGE, bool MEAS, unsigned STREAM, bool FEW = false>
__global__ __launch_bounds__(kBlock, sizeof(T) == 4 ? (MEAS ? 3 : 4) : GLACX_FP64_FLOW_WAVES) void flow_stage_kernel(
    const typename vec2<T>::type *__restrict__ win, typename vec2<T>::type *__restrict__ wout, T *__restrict__ acc,
    Geom g, T cz, T ca, double *__restrict__ meas)
{
    static_assert(!MEAS || (STAGE == 0 && sizeof(T) == 4),
                  "the measurement is fused into stage 0 only, FP64 has its own");
    __shared__ FlowLds<T> sh;
    const int mu = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // one direction per wavefront
    const int lane = threadIdx.x & 63;
    const int hb = flow_chunk(g, xcd_block(blockIdx.x, gridDim.x));
    const int h_raw = hb * (kFlowSites / 2) + (lane & 31);
    const bool valid = h_raw < g.vh;
    const int h = valid ? h_raw : g.vh - 1;  // idle lanes of a partial block mirror a real site, store nothing
    const int idx = parity_index(g, lane >> 5, h);
    const Site x = site_of(g, idx);
    // FP32: stages 1 and 2 read the link's accumulator now, so that its latency
    // passes under the staple loop instead of stalling the step after it; FP64 has
    // no registers left for it (with it in place early, 504 for 391 us)
    su3alg<T> cacc;
    if constexpr (STAGE != 0 && sizeof(T) == 4) cacc = acc_load<(STREAM & kStreamAcc) != 0>(acc, g, mu, idx);
    const DirView<T> vmu = dir_view<T>(win, g, mu);
    // the site's neighbours x + mu and x - mu, shared with the other
    // wavefronts, whose staples step the same way in direction mu
    __shared__ int nbr[2][4][kFlowSites];
    const Site xpm = site_step(g, x, mu, +1);
    const int ipm = xpm.idx, imm = site_step(g, x, mu, -1).idx;
    nbr[0][mu][lane] = ipm;
    nbr[1][mu][lane] = imm;
    lds_put(sh, mu, lane, load_link<T, R>(vmu, idx));
    lds_put(sh, 4 + mu, lane, load_link<T, R>(vmu, imm));
    T plaq = T(0);
    __syncthreads();
    auto back_link = [&](int d) -> M3<T> { return lds_get(sh, 4 + d, lane); };  // U_d(x - d)
    // FP64 plain stages: the x- and y-neighbours that are sites of this block, whose
    // own links are in LDS (with the block's sites in two whole runs of entries:
    // nearly every x-neighbour, and half the y-neighbours).  near_slot: such a
    // site's slot, -1 for the others; gather: the link, unless it is there;
    // take_near: the link, if it is.  These stages are bound by the lines a CU's L1
    // can have on their way at a time (load the links and multiply nothing, and
    // they take as long); this saves a fifth of the requests: 24^3 x 48 415 -> 391
    // and 387 -> 360 us.  The measuring stage has no registers for it (596 -> 645).
    constexpr bool kNear = sizeof(T) == 8 && !MEAS && !FEW;
    const bool near = kNear && (g.bh & 31) == 0;
    const int base0 = kNear ? parity_index(g, 0, hb * (kFlowSites / 2)) : 0, base1 = base0 + g.bh;
    auto near_slot = [&](bool xy, int at, bool same_parity) -> int {
        if (!near || !xy) return -1;
        const int p = (lane >> 5) ^ (same_parity ? 0 : 1), r = at - (p ? base1 : base0);
        return (unsigned)r < 32u ? p * 32 + r : -1;
    };
    auto gather = [&](const auto &d, int at, int slot) {
        return load_link_at(d, slot >= 0 ? kNoLink : tile_off(at));
    };
    auto take_near = [&](M3<T> &m, bool xy, int d, int slot) {
        if (near && xy) {
            const M3<T> n = lds_get(sh, d, slot >= 0 ? slot : lane);
#pragma unroll
            for (int e = 0; e < 9; e++) {
                m.e[e / 3][e % 3].r = slot >= 0 ? n.e[e / 3][e % 3].r : m.e[e / 3][e % 3].r;
                m.e[e / 3][e % 3].i = slot >= 0 ? n.e[e / 3][e % 3].i : m.e[e / 3][e % 3].i;
            }
        }
    };
    // staple A_mu(x) = sum_{nu != mu} [ U_nu(x+mu) U_mu(x+nu)^dag U_nu(x)^dag
    //                                 + U_nu(x+mu-nu)^dag U_mu(x-nu)^dag U_nu(x-nu) ]
    // (GLAC/actions/wilsongaugeaction.cpp:29-53)
    M3<T> a = zero3<T>();
    // measuring stage with three stored rows: T(U_mu(x) A_mu(x)) in compact form
    constexpr bool kCompactForce = MEAS && R == 3;
    T tz[8] = {T(0), T(0), T(0), T(0), T(0), T(0), T(0), T(0)};
    T held[2][8];  // measuring stage: see the end of a phase
    {
#pragma unroll 1
        for (int k = 0; k < 3; k++) {
            const int e = 3 * mu + k;
            // FP64 plain stages: the two wavefronts of a plane reach it together, so
            // that the upper links both of them gather come from L1 the second time
            // (24^3 x 48 440 -> 435 us).  FP32 sums the terms in another order, which
            // its results show in their last digits.
            const int nu = MEAS ? (int)((kPhaseNu >> (4 * e)) & 0xF)
                                : (sizeof(T) == 8 ? mu ^ (k + 1) : (mu + k + 1) & 3);
            const DirView<T> vnu = dir_view<T>(win, g, nu);
            const int ipn = nbr[0][nu][lane], imn = nbr[1][nu][lane];
            const int ipmmn = site_step(g, xpm, nu, -1).idx;
            if constexpr (MEAS) {
                // the same staple terms, kept apart for the clover leaves
                M3<T> up, low;
                const bool first = plane_first(mu, nu);
                const int d1 = first ? mu : nu, d2 = first ? nu : mu;
                const int slot = plane_slot(d1, d2);
                T f[8];
                if constexpr (R == 2) {
                    // SU(3) links (checked at upload): products from two rows,
                    // third rows rebuilt
                    M3<T> p;  // first two rows of U_nu(x+mu) U_mu(x+nu)^dag
                    mm<false, true, false, 2>(p, load_rows01<T, R>(vnu, ipm), load_link<T, R>(vmu, ipn));
                    mm<false, true, false, 2>(up, p, lds_get(sh, nu, lane));
                    rebuild_third_row(up);
                    const M3<T> q = su3_product<false>(load_rows01<T, R>(vmu, imn), load_link<T, R>(vnu, ipmmn));
                    mm<true, false, false>(low, q, back_link(nu));
                    add_to(a, up);
                    add_to(a, low);
                    const M3<T> u = lds_get(sh, mu, lane);
                    if (first) {
                        plaq += retrace_mul(u, up);
                        sub_from(up, low);
                        ta2_product<false>(u, up, f);
                    } else {
                        ta2_product<false>(u, low, f);
                    }
                } else {
                    // three stored rows may hold GLAC's det = -1 links: full
                    // products.  The upper term is finished (its leaf's
                    // plaquette and T(U_mu up)) before the lower one is
                    // formed, which keeps fewer matrices live: T(U_mu (up -
                    // low)) = T(U_mu up) - T(U_mu low).  The force needs only
                    // T(U_mu A) = sum of T(U_mu up) + T(U_mu low) over the
                    // terms, so it is accumulated in that compact form (8
                    // reals instead of the 3 x 3 staple sum).
                    mm<false, true, false>(up, mul_ad(load_link<T, R>(vnu, ipm), load_link<T, R>(vmu, ipn)),
                                           lds_get(sh, nu, lane));
                    T tu[8];
                    {
                        const M3<T> u = lds_get(sh, mu, lane);
                        if (first) plaq += retrace_mul(u, up);
                        ta2_product<false>(u, up, tu);
                    }
                    mm<false, false, false>(low, mul_dd(load_link<T, R>(vnu, ipmmn), load_link<T, R>(vmu, imn)),
                                            back_link(nu));
                    T fl[8];
                    ta2_product<false>(lds_get(sh, mu, lane), low, fl);
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        tz[j] += tu[j] + fl[j];
                        f[j] = first ? tu[j] - fl[j] : fl[j];
                    }
                }
                if ((kPhaseL3 >> e) & 1) {
                    // L3 = (U_d2(y) U_d1(x-d1))^dag (U_d1(y) U_d2(x-d2)),  y = x - d1 - d2
                    const int iy = site_step(g, site_step(g, x, d1, -1), d2, -1).idx;
                    const DirView<T> v1 = first ? vmu : vnu, v2 = first ? vnu : vmu;
                    T f3[8];
                    if constexpr (R == 2) {
                        const M3<T> m1 = su3_product<false>(load_rows01<T, R>(v1, iy), back_link(d2));
                        const M3<T> m2 = su3_product<false>(load_rows01<T, R>(v2, iy), back_link(d1));
                        ta2_product<true>(m2, m1, f3);
                    } else {
                        // L3 as a chain U_d1(x-d1)^dag U_d2(y)^dag U_d1(y) U_d2(x-d2):
                        // the same three products with one matrix live between them
                        M3<T> c1, c2;
                        mm<true, true, false>(c1, back_link(d1), load_link<T, R>(v2, iy));
                        mm<false, false, false>(c2, c1, load_link<T, R>(v1, iy));
                        mm<false, false, false>(c1, c2, back_link(d2));
                        ta2_of(c1, f3);
                    }
#pragma unroll
                    for (int j = 0; j < 8; j++) f[j] += f3[j];
                }
                // the plane's earlier contribution goes to its slot now, the later one
                // is held back and added once all the earlier ones are there
                if ((kPhaseAdd >> e) & 1) {
                    if (k == 1) {
#pragma unroll
                        for (int j = 0; j < 8; j++) held[0][j] = f[j];
                    } else {
#pragma unroll
                        for (int j = 0; j < 8; j++) held[1][j] = f[j];
                    }
                } else {
                    T(&fs)[8][kFlowSites] = flow_meas_lds<T>().f[slot];
#pragma unroll
                    for (int j = 0; j < 8; j++) fs[j][lane] = f[j];
                }
            } else if constexpr (R == 2) {
                // Two stored rows: form each SU(3) product's first two rows
                // from operands of which only those are needed, and rebuild
                // the product's third row once (36 multiply-adds fewer per
                // product than rebuilding both operands).
                M3<T> p;  // U_nu(x+mu) U_mu(x+nu)^dag, first two rows
                mm<false, true, false, 2>(p, load_rows01<T, R>(vnu, ipm), load_link<T, R>(vmu, ipn));
                // the upper term p U_nu(x)^dag is SU(3) too: its first two rows
                // need only p's, and its third is rebuilt from them
                M3<T> t;
                mm<false, true, false, 2>(t, p, lds_get(sh, nu, lane));
                rebuild_third_row(t);
                add_to(a, t);
                M3<T> q;  // U_mu(x-nu) U_nu(x+mu-nu), whose dagger the lower staple uses
                mm<false, false, false, 2>(q, load_rows01<T, R>(vmu, imn), load_link<T, R>(vnu, ipmmn));
                rebuild_third_row(q);
                mm<true, false, true>(a, q, back_link(nu));
            } else if constexpr (kNear) {
                // two waves per SIMD leave registers for all four gathers of the
                // term in flight at once (24^3 x 48 479 -> 454 us)
                const int sm = near_slot(mu < 2, ipm, false), sp = near_slot(nu < 2, ipn, false),
                          sn = near_slot(nu < 2, imn, false), sc = near_slot(mu < 2 && nu < 2, ipmmn, true);
                M3<T> u1 = gather(vnu, ipm, sm), u2 = gather(vmu, ipn, sp);
                M3<T> l1 = gather(vnu, ipmmn, sc), l2 = gather(vmu, imn, sn);
                __builtin_amdgcn_sched_barrier(0);
                take_near(u1, mu < 2, nu, sm);
                take_near(u2, nu < 2, mu, sp);
                mm<false, true, true>(a, mul_ad(u1, u2), lds_get(sh, nu, lane));
                take_near(l1, mu < 2 && nu < 2, nu, sc);
                take_near(l2, nu < 2, mu, sn);
                mm<false, false, true>(a, mul_dd(l1, l2), back_link(nu));
            } else {
                {
                    const M3<T> u1 = load_link<T, R>(vnu, ipm);
                    const M3<T> u2 = load_link<T, R>(vmu, ipn);
                    mm<false, true, true>(a, mul_ad(u1, u2), lds_get(sh, nu, lane));
                }
                {
                    const M3<T> u1 = load_link<T, R>(vnu, ipmmn);
                    const M3<T> u2 = load_link<T, R>(vmu, imn);
                    mm<false, false, true>(a, mul_dd(u1, u2), back_link(nu));
                }
            }
        }
    }
    if constexpr (MEAS) {
        __syncthreads();
#pragma unroll
        for (int k = 1; k < 3; k++) {
            const int e = 3 * mu + k, nu = (int)((kPhaseNu >> (4 * e)) & 0xF);
            if ((kPhaseAdd >> e) & 1) {
                T(&fs)[8][kFlowSites] =
                    flow_meas_lds<T>().f[plane_first(mu, nu) ? plane_slot(mu, nu) : plane_slot(nu, mu)];
#pragma unroll
                for (int j = 0; j < 8; j++) fs[j][lane] = fs[j][lane] + held[k - 1][j];
            }
        }
    }
    if constexpr (STAGE != 0 && sizeof(T) == 8) cacc = acc_load<(STREAM & kStreamAcc) != 0>(acc, g, mu, idx);
    if (valid) {
        const M3<T> u = lds_get(sh, mu, lane);
        su3alg<T> z;
        if constexpr (kCompactForce) {
            z = force_from_ta2(tz);
        } else {
            z = force_from_omega(mul(u, a));
        }
        finish_link<T, R, STAGE, STREAM>(wout, acc, g, mu, idx, u, z, cacc, cz, ca);
    }
    if constexpr (MEAS) {
        // every lane is a real site here (the launch requires whole chunks)
        __syncthreads();
        T fa[8], fb[8];
        if (mu < 3) {
#pragma unroll
            for (int k = 0; k < 8; k++) {
                fa[k] = flow_meas_lds<T>().f[mu][k][lane];
                fb[k] = flow_meas_lds<T>().f[mu + 3][k][lane];
            }
        }
        measure_block<T>(g, hb, mu, plaq, fa, fb, meas);
    }
}

// ---- measuring stage of FP64 links --------------------------------------------
// FP64 has the registers to keep all three of a wavefront's contributions to F (48)
// until the end, so nothing waits between the terms, and they are handed over in the
// LDS of the shared links, which nobody needs any more by then.  The six planes'
// slots of the kernel above would leave no room at two blocks per CU to share the
// backward links; without them it is 68 link gathers per site for 88, and the
// gathers are what bounds FP64 stages.
//
// 24^3 x 48: 529 us, where the kernel above (backward links gathered, a barrier after
// each phase) took 600; the phases with both planes of a pair at a time, slots
// for those and three shared backward links 585.  More gathers in flight or
// x- and y-neighbours from LDS gain nothing here (516 to 557).
struct Measure64Lds {
    union {
        LdsMats<double, 8> sh;               // U_mu(x), then U_mu(x - mu)
        double part[2][6][8][kFlowSites];    // F of a plane: its first wavefront's part, its second's
    };
};

template <unsigned STREAM>
__global__ __launch_bounds__(kBlock, 2) void flow_measure64_kernel(const double2 *__restrict__ win,
                                                                   double2 *__restrict__ wout, double *__restrict__ acc,
                                                                   Geom g, double cz, double *__restrict__ meas)
{
    using T = double;
    constexpr int R = 3;
    __shared__ __align__(16) Measure64Lds lds;
    __shared__ int nbr[2][4][kFlowSites];
    const int mu = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int hb = flow_chunk(g, xcd_block(blockIdx.x, gridDim.x));
    // every lane is a real site (the launch requires whole chunks)
    const int idx = parity_index(g, lane >> 5, hb * (kFlowSites / 2) + (lane & 31));
    const Site x = site_of(g, idx);
    const DirView<T> vmu = dir_view<T>(win, g, mu);
    const Site xpm = site_step(g, x, mu, +1);
    const int ipm = xpm.idx, imm = site_step(g, x, mu, -1).idx;
    nbr[0][mu][lane] = ipm;
    nbr[1][mu][lane] = imm;
    lds_put(lds.sh, mu, lane, load_link<T, R>(vmu, idx));
    lds_put(lds.sh, 4 + mu, lane, load_link<T, R>(vmu, imm));
    __syncthreads();
    T plaq = 0, tz[8] = {0, 0, 0, 0, 0, 0, 0, 0};  // tz: T(U_mu(x) A_mu(x)), as above
    T f[3][8];
    // form() keeps the loads of the next product behind the one before (200 to 230
    // registers; free to move them the compiler spills)
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const int e = 3 * mu + k, nu = (int)((kPhaseNu >> (4 * e)) & 0xF);
        const bool first = plane_first(mu, nu);
        const DirView<T> vnu = dir_view<T>(win, g, nu);
        const int ipn = nbr[0][nu][lane], imn = nbr[1][nu][lane];
        const int ipmmn = site_step(g, xpm, nu, -1).idx;
        {
            M3<T> up, low;
            M3<T> p = mul_ad(load_link<T, R>(vnu, ipm), load_link<T, R>(vmu, ipn));
            form(p);
            mm<false, true, false>(up, p, lds_get(lds.sh, nu, lane));
            form(up);
            T tu[8], fl[8];
            {
                const M3<T> u = lds_get(lds.sh, mu, lane);
                if (first) plaq += retrace_mul(u, up);
                ta2_product<false>(u, up, tu);
                form(tu);
            }
            p = mul_dd(load_link<T, R>(vnu, ipmmn), load_link<T, R>(vmu, imn));
            form(p);
            mm<false, false, false>(low, p, lds_get(lds.sh, 4 + nu, lane));
            form(low);
            ta2_product<false>(lds_get(lds.sh, mu, lane), low, fl);
#pragma unroll
            for (int j = 0; j < 8; j++) {
                tz[j] += tu[j] + fl[j];
                f[k][j] = first ? tu[j] - fl[j] : fl[j];
            }
        }
        if ((kPhaseL3 >> e) & 1) {
            const int d1 = first ? mu : nu, d2 = first ? nu : mu;
            const int iy = site_step(g, site_step(g, x, d1, -1), d2, -1).idx;
            const DirView<T> v1 = first ? vmu : vnu, v2 = first ? vnu : vmu;
            M3<T> c1, c2;
            mm<true, true, false>(c1, lds_get(lds.sh, 4 + d1, lane), load_link<T, R>(v2, iy));
            form(c1);
            mm<false, false, false>(c2, c1, load_link<T, R>(v1, iy));
            form(c2);
            mm<false, false, false>(c1, c2, lds_get(lds.sh, 4 + d2, lane));
            T f3[8];
            ta2_of(c1, f3);
#pragma unroll
            for (int j = 0; j < 8; j++) f[k][j] += f3[j];
        }
        form(f[k]);
        form(tz);
    }
    const su3alg<T> z = force_from_ta2(tz);
    finish_link<T, R, 0, STREAM>(wout, acc, g, mu, idx, lds_get(lds.sh, mu, lane), z, z, cz, 0.0);
    __syncthreads();  // the shared links are done with
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const int nu = (int)((kPhaseNu >> (4 * (3 * mu + k))) & 0xF);
        const bool first = plane_first(mu, nu);
        T(&o)[8][kFlowSites] = lds.part[first ? 0 : 1][first ? plane_slot(mu, nu) : plane_slot(nu, mu)];
#pragma unroll
        for (int j = 0; j < 8; j++) o[j][lane] = f[k][j];
    }
    __syncthreads();
    T fa[8], fb[8];
    if (mu < 3) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            fa[j] = lds.part[0][mu][j][lane] + lds.part[1][mu][j][lane];
            fb[j] = lds.part[0][mu + 3][j][lane] + lds.part[1][mu + 3][j][lane];
        }
    }
    measure_block<T>(g, hb, mu, plaq, fa, fb, meas);
}

// ---- measuring stage of a small lattice ----------------------------------------
// Where the blocks do not fill the chip, the kernels above are four wavefronts
// alone on their SIMDs, and their time the chain of three phases, each two gathers
// and five to eight products.  Here a block has twelve wavefronts:
// wavefront (mu, k) works out mu's phase k by itself, gathering the links that the
// kernels above share; those of k = 1, 2 leave their part of the force in LDS, and
// (mu, 0) adds the parts in the phases' order and finishes the link.  F's two
// contributions per plane stand side by side instead of the later one being
// added to the earlier.  The same sums as above.
//
// What bounds it: a launch and the chain gathers, products, force, exponential
// (at 4^4 it takes hardly less than at 8^3 x 16).  Microseconds with 2 of event
// timing, the kernels above and this one, compressed FP32, FP32 and FP64:
//     64 blocks    14.2 11.2    15.6 12.5    17.5 16.9
//    256 blocks    14.7 12.1    16.5 13.6    18.5 18.6
//    768 blocks    19.7 28.9    23.8 33.7    40.5 52.1
// For the plain stages, whose four wavefronts hold no phases, the same split gains
// 0.6 us of 8.3 (compressed FP32) and nothing otherwise, so they have none.
constexpr int kWideBlocks = 256;  // one block of twelve wavefronts per CU

template <class T, int R> struct WideLds {
    using V2 = typename vec2<T>::type;
    V2 mat[R == 2 ? 4 : 1][4][R == 2 ? 9 : 1][R == 2 ? 64 : 1];  // two stored rows: a phase's two staple terms
    T part[2][4][R == 2 ? 1 : 9][64];                           // plaquette; three: also T(U_mu (up + low))
    T f[2][6][8][64];                                           // F of a plane: the earlier phase's part, the later's
};

template <class T, class V2> __device__ __forceinline__ void wide_put(V2 (&s)[9][64], int lane, const M3<T> &m)
{
#pragma unroll
    for (int e = 0; e < 9; e++) {
        V2 z;
        z.x = m.e[e / 3][e % 3].r;
        z.y = m.e[e / 3][e % 3].i;
        s[e][lane] = z;
    }
}
template <class T, class V2> __device__ __forceinline__ M3<T> wide_get(const V2 (&s)[9][64], int lane)
{
    M3<T> m;
#pragma unroll
    for (int e = 0; e < 9; e++) m.e[e / 3][e % 3] = {s[e][lane].x, s[e][lane].y};
    return m;
}

template <class T, int R>
__global__ __launch_bounds__(3 * kBlock, 3) void flow_measure_wide_kernel(
    const typename vec2<T>::type *__restrict__ win, typename vec2<T>::type *__restrict__ wout, T *__restrict__ acc,
    Geom g, T cz, double *__restrict__ meas)
{
    __shared__ __align__(16) WideLds<T, R> lds;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), mu = wave & 3, k = wave >> 2;
    const int lane = threadIdx.x & 63;
    const int hb = flow_chunk(g, xcd_block(blockIdx.x, gridDim.x));
    // every lane is a real site (the launch requires whole chunks)
    const int idx = parity_index(g, lane >> 5, hb * (kFlowSites / 2) + (lane & 31));
    const Site x = site_of(g, idx);
    const int e = 3 * mu + k, nu = (int)((kPhaseNu >> (4 * e)) & 0xF);
    const bool first = plane_first(mu, nu);
    const int d1 = first ? mu : nu, d2 = first ? nu : mu;
    const DirView<T> vmu = dir_view<T>(win, g, mu), vnu = dir_view<T>(win, g, nu);
    const Site xpm = site_step(g, x, mu, +1);
    const int ipm = xpm.idx, ipn = site_step(g, x, nu, +1).idx, imn = site_step(g, x, nu, -1).idx;
    const int ipmmn = site_step(g, xpm, nu, -1).idx;
    T plaq = T(0), f[8], tz[8];
    M3<T> a = zero3<T>();
    {
        // the phase's staple terms and their part of F, as above
        M3<T> up, low;
        if constexpr (R == 2) {
            M3<T> p;
            mm<false, true, false, 2>(p, load_rows01<T, R>(vnu, ipm), load_link<T, R>(vmu, ipn));
            mm<false, true, false, 2>(up, p, load_link<T, R>(vnu, idx));
            rebuild_third_row(up);
            const M3<T> q = su3_product<false>(load_rows01<T, R>(vmu, imn), load_link<T, R>(vnu, ipmmn));
            mm<true, false, false>(low, q, load_link<T, R>(vnu, imn));
            if (k > 0) {
                wide_put(lds.mat[2 * (k - 1)][mu], lane, up);
                wide_put(lds.mat[2 * (k - 1) + 1][mu], lane, low);
            } else {
                add_to(a, up);
                add_to(a, low);
            }
            const M3<T> u = load_link<T, R>(vmu, idx);
            if (first) {
                plaq = retrace_mul(u, up);
                sub_from(up, low);
                ta2_product<false>(u, up, f);
            } else {
                ta2_product<false>(u, low, f);
            }
        } else {
            T tu[8], fl[8];
            {
                M3<T> p = mul_ad(load_link<T, R>(vnu, ipm), load_link<T, R>(vmu, ipn));
                form(p);
                mm<false, true, false>(up, p, load_link<T, R>(vnu, idx));
                form(up);
                const M3<T> u = load_link<T, R>(vmu, idx);
                if (first) plaq = retrace_mul(u, up);
                ta2_product<false>(u, up, tu);
                form(tu);
            }
            {
                M3<T> p = mul_dd(load_link<T, R>(vnu, ipmmn), load_link<T, R>(vmu, imn));
                form(p);
                mm<false, false, false>(low, p, load_link<T, R>(vnu, imn));
                form(low);
                ta2_product<false>(load_link<T, R>(vmu, idx), low, fl);
                form(fl);
            }
#pragma unroll
            for (int j = 0; j < 8; j++) {
                tz[j] = tu[j] + fl[j];
                f[j] = first ? tu[j] - fl[j] : fl[j];
            }
            if (k > 0) {
#pragma unroll
                for (int j = 0; j < 8; j++) lds.part[k - 1][mu][1 + j][lane] = tz[j];
            }
        }
        if (k > 0) lds.part[k - 1][mu][0][lane] = plaq;
    }
    if ((kPhaseL3 >> e) & 1) {
        const Site xm1 = site_step(g, x, d1, -1);
        const int i1 = xm1.idx, i2 = site_step(g, x, d2, -1).idx, iy = site_step(g, xm1, d2, -1).idx;
        const DirView<T> v1 = first ? vmu : vnu, v2 = first ? vnu : vmu;
        T f3[8];
        if constexpr (R == 2) {
            const M3<T> m1 = su3_product<false>(load_rows01<T, R>(v1, iy), load_link<T, R>(v2, i2));
            const M3<T> m2 = su3_product<false>(load_rows01<T, R>(v2, iy), load_link<T, R>(v1, i1));
            ta2_product<true>(m2, m1, f3);
        } else {
            M3<T> c1, c2;
            mm<true, true, false>(c1, load_link<T, R>(v1, i1), load_link<T, R>(v2, iy));
            form(c1);
            mm<false, false, false>(c2, c1, load_link<T, R>(v1, iy));
            form(c2);
            mm<false, false, false>(c1, c2, load_link<T, R>(v2, i2));
            ta2_of(c1, f3);
        }
#pragma unroll
        for (int j = 0; j < 8; j++) f[j] += f3[j];
    }
    T(&fs)[8][64] = lds.f[(kPhaseAdd >> e) & 1][plane_slot(d1, d2)];
#pragma unroll
    for (int j = 0; j < 8; j++) fs[j][lane] = f[j];
    __syncthreads();
    if (k > 0) {
        __syncthreads();  // measure_block's
        return;
    }
    const M3<T> u = load_link<T, R>(vmu, idx);
    su3alg<T> z;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        plaq += lds.part[h][mu][0][lane];
        if constexpr (R == 2) {
            add_to(a, wide_get<T>(lds.mat[2 * h][mu], lane));
            add_to(a, wide_get<T>(lds.mat[2 * h + 1][mu], lane));
        } else {
#pragma unroll
            for (int j = 0; j < 8; j++) tz[j] += lds.part[h][mu][1 + j][lane];
        }
    }
    if constexpr (R == 2)
        z = force_from_omega(mul(u, a));
    else
        z = force_from_ta2(tz);
    // streaming both: the fields are below 18 MiB
    finish_link<T, R, 0, kStreamAcc | kStreamLinks>(wout, acc, g, mu, idx, u, z, z, cz, T(0));
    T fa[8], fb[8];
    if (mu < 3) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            fa[j] = lds.f[0][mu][j][lane] + lds.f[1][mu][j][lane];
            fb[j] = lds.f[0][mu + 3][j][lane] + lds.f[1][mu + 3][j][lane];
        }
    }
    measure_block<T>(g, hb, mu, plaq, fa, fb, meas);
}

// Dynamic LDS reserved per block; nonzero values cap the blocks resident per
// CU (a tuning parameter of the launch, set at build time).
#ifndef GLACX_FLOW_LDS_BYTES
#define GLACX_FLOW_LDS_BYTES 0
#endif

// Fusing the measurement needs each block's 32 sites per parity to be one
// chunk of one run (a single time slice): run % 32 == 0, which holds for
// every lattice with bz Ny Nx / 2 divisible by 32.
bool flow_measure_fusable(const Geom &g) { return g.run % (kFlowSites / 2) == 0; }

template <class T, int R, unsigned STREAM, bool FEW>
static void launch_stage(const void *win, void *wout, void *acc, const Geom &g, int stage, double eps, double *meas,
                         hipStream_t s)
{
    using V2 = typename vec2<T>::type;
    const unsigned blocks = (unsigned)((g.vh + kFlowSites / 2 - 1) / (kFlowSites / 2));
    const V2 *in = (const V2 *)win;
    V2 *out = (V2 *)wout;
    T *a = (T *)acc;
    switch (stage) {
    case 0:
        if (meas) {
            if (blocks <= kWideBlocks)
                flow_measure_wide_kernel<T, R><<<blocks, 3 * kBlock, 0, s>>>(in, out, a, g, T(0.25 * eps), meas);
            else if constexpr (sizeof(T) == 8)
                flow_measure64_kernel<STREAM><<<blocks, kBlock, 0, s>>>(in, out, a, g, T(0.25 * eps), meas);
            else
                flow_stage_kernel<T, R, 0, true, STREAM>
                    <<<blocks, kBlock, GLACX_FLOW_LDS_BYTES, s>>>(in, out, a, g, T(0.25 * eps), T(0), meas);
            break;
        }
        flow_stage_kernel<T, R, 0, false, STREAM, FEW>
            <<<blocks, kBlock, GLACX_FLOW_LDS_BYTES, s>>>(in, out, a, g, T(0.25 * eps), T(0), nullptr);
        break;
    case 1:
        flow_stage_kernel<T, R, 1, false, STREAM, FEW><<<blocks, kBlock, GLACX_FLOW_LDS_BYTES, s>>>(
            in, out, a, g, T(8.0 / 9.0 * eps), T(17.0 / 36.0 * eps), nullptr);
        break;
    default:
        flow_stage_kernel<T, R, 2, false, STREAM, FEW>
            <<<blocks, kBlock, GLACX_FLOW_LDS_BYTES, s>>>(in, out, a, g, T(0.75 * eps), T(1), nullptr);
        break;
    }
}

template <class T, int R>
void launch_flow_stage(const void *win, void *wout, void *acc, const Geom &g, int stage, double eps, double *meas,
                       hipStream_t s)
{
    // the table at StreamBits
    const size_t fields = (size_t)2 * 4 * g.v * 6 * R * sizeof(T), accumulator = (size_t)32 * g.v * sizeof(T);
    constexpr size_t kInfinityCache = (size_t)256 << 20;
    constexpr size_t kL2 = (size_t)(sizeof(T) == 8 ? 16 : 28) << 20;
    constexpr unsigned kBoth = kStreamAcc | kStreamLinks;
    if constexpr (sizeof(T) == 8) {
        if (g.vh <= kFewBlocks * (kFlowSites / 2)) {  // the table at kFewBlocks
            if (fields < kL2)
                launch_stage<T, R, kBoth, true>(win, wout, acc, g, stage, eps, meas, s);
            else
                launch_stage<T, R, 0, true>(win, wout, acc, g, stage, eps, meas, s);
            return;
        }
    } else if (fields < kL2) {
        launch_stage<T, R, kBoth, false>(win, wout, acc, g, stage, eps, meas, s);
        return;
    }
    if (fields > kInfinityCache)
        launch_stage<T, R, kBoth, false>(win, wout, acc, g, stage, eps, meas, s);
    else if (fields + accumulator >= kInfinityCache)
        launch_stage<T, R, kStreamAcc, false>(win, wout, acc, g, stage, eps, meas, s);
    else
        launch_stage<T, R, 0, false>(win, wout, acc, g, stage, eps, meas, s);
}

template void launch_flow_stage<float, 3>(const void *, void *, void *, const Geom &, int, double, double *,
                                         hipStream_t);
template void launch_flow_stage<float, 2>(const void *, void *, void *, const Geom &, int, double, double *,
                                         hipStream_t);
template void launch_flow_stage<double, 3>(const void *, void *, void *, const Geom &, int, double, double *,
                                          hipStream_t);

} // namespace glacx
