// kernels.hpp -- host-side launchers of the gfx950 kernels (one translation
// unit per kernel family) and the shared block reduction.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "lattice.hpp"

namespace glacx {

constexpr int kBlock = 256;  // 4 wavefronts of 64

// Flow-stage launch shape: a block covers 64 consecutive sites, wavefront w
// handling direction mu = w, so the four links of a site share a CU.
constexpr int kFlowSites = 64;

struct MetroParams {
    double beta;
    double eps;
    int n_hit;
    int reunit;
    uint64_t seed;
    uint64_t sweep;
};

// Sum `N` per-thread doubles over a block of WAVES wavefronts; thread 0 gets
// the sums.  Wavefront shuffle, then one LDS exchange between the wavefronts;
// the order of additions is fixed, so results are reproducible run to run.
template <int N, int WAVES = kBlock / 64> __device__ __forceinline__ void block_sum(double (&v)[N])
{
    __shared__ double lds[N][WAVES];
#pragma unroll
    for (int k = 0; k < N; k++) {
        double x = v[k];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
        v[k] = x;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < N; k++) lds[k][wave] = v[k];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < N; k++) {
            double s = lds[k][0];
#pragma unroll
            for (int w = 1; w < WAVES; w++) s += lds[k][w];
            v[k] = s;
        }
    }
}

// ---- launchers (explicitly instantiated for float and double) ------------
template <class T, int R> void launch_pack(const double *stage, void *f, const Geom &g, int site_major, hipStream_t s);
template <class T, int R> void launch_unpack(const void *f, double *stage, const Geom &g, int site_major, hipStream_t s);
// *flag = 1 when one of n links (18 doubles each) is not within `bound` of SU(3)
// (see su3_check_kernel); otherwise left as it is.
void launch_su3_check(const double *links, int n, double bound, int *flag, hipStream_t s);
// Hot-start kinds (the values of the C ABI's GLACX_HOT_*).
enum HotKind { HOT_HAAR = 0, HOT_GLAC_RANDOM = 1, HOT_RST = 2 };
template <class T, int R> void launch_hot_start(void *f, const Geom &g, uint64_t seed, int kind, double eps, hipStream_t s);
template <class T, int R> void launch_cold_start(void *f, const Geom &g, hipStream_t s);
template <class T, int R>
void launch_action_derivative(const void *f, double *stage, const Geom &g, int mu, hipStream_t s);

// Clover measurement partials: kMeasAcc doubles {plaq, E, q, w} per
// (chunk, t) slot, chunk c of time slice t at partials[kMeasAcc (c Nt + t)]
// (w, the Weinberg density, only in the SuperSampler variant).
constexpr int kMeasAcc = 4;

// Clover measurement: per-block partial sums, then a fixed-order reduction of
// `rows` measurements (measure_partials_count(g) doubles of partials each, side
// by side) into rows of out, `pitch` doubles apart: {plaq, E_raw, Q, Q(t)...},
// or with `super` (GLAC's SuperSampler) {plaq, E_raw, Q, W, Q(t)..., W(t)...}.
// mode: 0 plain, 1 SuperSampler (Weinberg), 2 plain plus per-site densities into
// density[0..V) (charge) and density[V..2V) (action), GLAC site order.
int measure_partials_count(const Geom &g);
template <class T, int R>
void launch_measure(const void *f, const Geom &g, double *partials, int mode, double *density, hipStream_t s);
void launch_measure_finish(double *partials, const Geom &g, double *out, bool super, int rows, size_t pitch,
                           hipStream_t s);

int plaquette_partials_count(const Geom &g);
template <class T, int R> void launch_plaquette(const void *f, const Geom &g, double *partials, hipStream_t s);
void launch_plaquette_finish(const double *partials, int nparts, const Geom &g, double *out, int rows, hipStream_t s);

// One RK3 stage (0, 1, 2): win -> wout, accumulator read/written in acc.
// With `meas` (stage 0 only, flow_measure_fusable(g)) the stage also writes the
// clover-measurement partials of win into meas, in the layout launch_measure_finish
// reads.
template <class T, int R>
void launch_flow_stage(const void *win, void *wout, void *acc, const Geom &g, int stage, double eps, double *meas,
                       hipStream_t s);
bool flow_measure_fusable(const Geom &g);

// Accepted hits of a sweep are counted in kCountSlots slots, wavefront w's (or block
// w's, in small lattices) in slot w % kCountSlots: on one address the blocks of a small
// lattice, which end together, queue for 5 of their 18 us (512 blocks).  launch_count_sum adds up
// `sweeps` sweeps' slots and leaves them cleared.
constexpr int kCountSlots = 256;
__device__ __forceinline__ int count_slot(unsigned block) { return (int)(block & (kCountSlots - 1)); }
// The wavefront's accepted hits into its slot.
__device__ __forceinline__ void add_count(unsigned long long *count, unsigned wavefront, int n)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) n += __shfl_down(n, off, 64);
    if ((threadIdx.x & 63) == 0) atomicAdd(count + count_slot(wavefront), (unsigned long long)n);
}
void launch_count_sum(unsigned long long *slots, unsigned long long *counts, int sweeps, hipStream_t s);

// One checkerboard sub-sweep (mu, parity), in place; accepted hits are added
// to the sweep's slots at `count`.
template <class T, int R>
void launch_metropolis(void *f, const Geom &g, int mu, int parity, const MetroParams &p,
                       unsigned long long *count, hipStream_t s);

// ---- learned proposal (k_learned.hip) ----------------------------------------
// Samples are 36 reals (A then U, 18 each) in nine float4 planes: reals
// 4q..4q+3 of sample s at (float4 *)out + q * cap + s.
template <class T, int R>
void launch_collect(const void *f, const Geom &g, int mu, int parity, int stride, float *out, size_t cap, size_t base,
                    hipStream_t s);
int feature_moments_blocks(size_t n);
void launch_feature_moments(const float *smp, size_t cap, size_t n, double beta, double *partials, float *mean_std,
                            hipStream_t s);
// One training step over `batch` samples (drawn from the first n_samples, or
// the first `batch` in order with draws read from zin when zin != nullptr);
// adam_t > 0 applies an Adam update (bias corrections for step adam_t).
// inter: train_inter_floats(batch) floats; loss_partials: train_groups(batch)
// doubles; the step's loss goes to *loss.
size_t train_inter_floats(int batch);
int train_groups(int batch);
void launch_train_step(const float *smp, size_t cap, size_t n_samples, int batch, int draws, uint64_t seed,
                       uint64_t step, double beta, float *params, const float *mean_std, const float *zin,
                       float *inter, double *loss_partials, double *loss, float *grad, float *m, float *v, float lr,
                       int adam_t, unsigned short *bf16, hipStream_t s);
void launch_to_bf16(const float *params, unsigned short *bf16, hipStream_t s);
template <class T, int R>
void launch_metropolis_learned(void *f, const Geom &g, int mu, int parity, const MetroParams &p,
                               const unsigned short *wbf16, const float *mean_std, unsigned long long *count,
                               hipStream_t s);
void launch_proposal_eval(const float *feat, int n, const unsigned short *wbf16, const float *mean_std, float *out,
                          int *ok, hipStream_t s);
constexpr int kProposalParams = 2468;

} // namespace glacx
