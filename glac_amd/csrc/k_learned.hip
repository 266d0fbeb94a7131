// k_learned.hip -- training and sampling kernels of the learned proposal
// (definitions in learned.hpp; no GLAC counterpart).
//
// Training data: (staple A, link U) pairs read off the chain of the plain
// sampler.  Objective, per sample and per draw z (W = U A, w = L(A) z,
// Y = i w.lambda / 2):
//     dS_2 = -(beta / 3) (Re tr(Y W) + Re tr(Y Y W) / 2),  alpha = min(1, e^{-dS_2}),
//     loss = -alpha |w|^2              (negative expected squared jump distance).
// The second-order dS only shapes the proposal; the sampler uses the exact
// exponential and exact dS.
//
// A training step is two kernels: train_kernel (one wavefront per 16 samples:
// forward, loss and back-propagation to the layer inputs, the layers on the
// matrix cores) and update_kernel (the batch sums of the outer products on the
// FP64 matrix cores, then Adam).  Both keep every sum in the order of a plain
// loop: a training run amplifies a last-bit change of a gradient to per cent
// within 200 steps.
#include <algorithm>

#include "kernels.hpp"
#include "learned.hpp"
#include "proposal.hpp"

namespace glacx {

// Samples hold 36 reals: A (18) then U (18), as nine float4 planes (reals
// 4q..4q+3 of sample s at plane q): collection writes and the moments read
// them coalesced, and a training step's random samples touch nine cache lines
// each instead of 36.
//
// Per-sample columns kept for the gradient: x, h1, h2, do, da2, da1 and a
// column of ones (the input of the biases).
constexpr int kColX = 0, kColH1 = kColX + kMlpIn, kColH2 = kColH1 + kMlpH1, kColDo = kColH2 + kMlpH2,
              kColDa2 = kColDo + kMlpOut, kColDa1 = kColDa2 + kMlpH2, kColOne = kColDa1 + kMlpH1, kCols = kColOne + 1;

// reals [0, 18) (A) or [0, 36) (A and U) of sample i
template <int N> __device__ __forceinline__ void read_sample(const float4 *__restrict__ smp, size_t cap, size_t i,
                                                             float v[4 * N])
{
#pragma unroll
    for (int q = 0; q < N; q++) {
        const float4 t = smp[(size_t)q * cap + i];
        v[4 * q] = t.x, v[4 * q + 1] = t.y, v[4 * q + 2] = t.z, v[4 * q + 3] = t.w;
    }
}
__device__ __forceinline__ M3<float> matrix_of(const float *v)
{
    M3<float> m;
#pragma unroll
    for (int k = 0; k < 9; k++) m.e[k / 3][k % 3] = {v[2 * k], v[2 * k + 1]};
    return m;
}

// ---- sample collection -----------------------------------------------------
template <class T, int R>
__global__ __launch_bounds__(kBlock) void collect_kernel(const typename vec2<T>::type *__restrict__ f, Geom g, int mu,
                                                         int parity, int stride, float4 *__restrict__ out, size_t cap,
                                                         size_t base)
{
    const int h = (blockIdx.x * kBlock + threadIdx.x) * stride;
    if (h >= g.vh) return;
    const size_t s = base + (size_t)(h / stride);
    if (s >= cap) return;
    const int idx = parity_index(g, parity, h);
    const Site x = site_of(g, idx);
    const M3<T> a = staple<T, R>(f, g, x, mu);
    const M3<T> u = load_link<T, R>(f, g, mu, idx);
    float v[36];
#pragma unroll
    for (int k = 0; k < 9; k++) {
        v[2 * k] = float(a.e[k / 3][k % 3].r);
        v[2 * k + 1] = float(a.e[k / 3][k % 3].i);
        v[18 + 2 * k] = float(u.e[k / 3][k % 3].r);
        v[18 + 2 * k + 1] = float(u.e[k / 3][k % 3].i);
    }
#pragma unroll
    for (int q = 0; q < 9; q++)
        out[(size_t)q * cap + s] = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
}

// ---- feature standardisation ---------------------------------------------------
// Sums of the six features and their squares: at most kMomentBlocks blocks
// stride over the samples, so that the second kernel's sum stays short
// whatever the sample count (one thread summing a partial per 256 samples took
// 646 us for 262 144 samples, beside the first kernel's 12 us; now 4.7 us).
constexpr int kMomentBlocks = 1024;

__global__ __launch_bounds__(kBlock) void feature_moments_kernel(const float4 *__restrict__ smp, size_t cap, size_t n,
                                                                 double beta, double *__restrict__ partials)
{
    double acc[12];
#pragma unroll
    for (int k = 0; k < 12; k++) acc[k] = 0.0;
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock) {
        float fe[6], v[20];
        read_sample<5>(smp, cap, i, v);
        staple_features(matrix_of(v), beta, fe);
#pragma unroll
        for (int k = 0; k < 6; k++) {
            acc[k] += fe[k];
            acc[6 + k] += (double)fe[k] * fe[k];
        }
    }
    block_sum<12>(acc);
    if (threadIdx.x == 0)
        for (int k = 0; k < 12; k++) partials[(size_t)blockIdx.x * 12 + k] = acc[k];
}

// One block: thread (group, k) sums every kMomentGroups-th partial of moment
// k, then one thread per feature adds the groups, both in a fixed order.
constexpr int kMomentGroups = kBlock / 12;

__global__ __launch_bounds__(kBlock) void feature_moments_finish(const double *__restrict__ partials, int nblk,
                                                                 size_t n, float *__restrict__ mean_std)
{
    __shared__ double sums[kMomentGroups][12];
    const int group = threadIdx.x / 12, m = threadIdx.x - 12 * group;
    if (group < kMomentGroups) {
        double s = 0.0;
#pragma unroll 8
        for (int b = group; b < nblk; b += kMomentGroups) s += partials[(size_t)b * 12 + m];
        sums[group][m] = s;
    }
    __syncthreads();
    const int k = threadIdx.x;
    if (k >= 6) return;
    double s = 0.0, s2 = 0.0;
    for (int b = 0; b < kMomentGroups; b++) {
        s += sums[b][k];
        s2 += sums[b][6 + k];
    }
    const double mean = s / (double)n;
    const double var = s2 / (double)n - mean * mean;
    mean_std[k] = (float)mean;
    mean_std[6 + k] = (float)(var > 1e-12 ? sqrt(var) : 1.0);
}

// ---- training step -------------------------------------------------------------
// One wavefront (a block of its own) trains on 16 samples.  Lane l works for
// sample l % 16 and, in slot l / 16, on every fourth draw and a quarter of the
// Cholesky factor's entries; the network's layers are FP32 matrix products
// [units x inputs] [inputs x 16 samples] on v_mfma_f32_16x16x4 (weights as the
// A operand), whose columns pass through LDS from layer to layer.  The matrix
// instruction adds its four products one after the other with one rounding
// each (checked on random and denormal operands), so a layer rounds exactly as
// a loop of fused multiply-adds over its inputs.
//
// What bounds it: latency.  The default batch of 4096 is 256 wavefronts, one
// per CU, each a chain sample -> features -> layers -> draws -> backward.
// One thread per sample with all layers in its registers (64 wavefronts) took
// 39 us a step at batch 4096 with 4 draws, 16 us now; four wavefronts per
// 64 samples with the weights in scalar registers 55 us (they spill).
constexpr int kTrainSites = 16;
constexpr int kColStride = 20;  // words per column in LDS: a tile's results go to 64 different banks

struct TrainLds {
    float col[kCols][kColStride];     // the gradient's columns
    float dz[4][16][kTrainSites];     // per slot: d loss / d w (8) and z (8) of its draw
};

// Row and column of the Cholesky factor behind output e (eight diagonal
// entries, then the rows below them): the two indices packed as 16 a + b.
__device__ constexpr unsigned char kCholIndex[kMlpOut] = {
    0x00, 0x11, 0x22, 0x33, 0x44, 0x55, 0x66, 0x77, 0x10, 0x20, 0x21, 0x30, 0x31, 0x32, 0x40, 0x41, 0x42, 0x43,
    0x50, 0x51, 0x52, 0x53, 0x54, 0x60, 0x61, 0x62, 0x63, 0x64, 0x65, 0x70, 0x71, 0x72, 0x73, 0x74, 0x75, 0x76};

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__global__ __launch_bounds__(64, 1) void train_kernel(const float4 *__restrict__ smp, size_t cap, size_t n_samples,
                                                      int batch, int draws, uint64_t seed, uint64_t step, double beta,
                                                      const float *__restrict__ P, const float *__restrict__ mean_std,
                                                      const float *__restrict__ zin, float *__restrict__ inter,
                                                      double *__restrict__ loss_partials)
{
    __shared__ TrainLds lds;
    const int lane = threadIdx.x, j = lane & 15, slot = lane >> 4;
    const int i_raw = blockIdx.x * kTrainSites + j;
    const bool valid = i_raw < batch;
    const int i = valid ? i_raw : batch - 1;  // idle columns mirror a real sample, with zero derivatives
    size_t s;
    if (zin) {
        s = (size_t)i;
    } else {
        uint32_t c[4] = {(uint32_t)i, (uint32_t)(step >> 32), (uint32_t)step, 0x7E57u};
        philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
        s = (size_t)((((uint64_t)c[0] << 32) | c[1]) % n_samples);
    }
    float v36[36];
    read_sample<9>(smp, cap, s, v36);
    const M3<float> A = matrix_of(v36), U = matrix_of(v36 + 18);
    {
        float fe[6], x[8];
        staple_features(A, beta, fe);
#pragma unroll
        for (int k = 0; k < kMlpIn; k++) x[k] = (fe[k] - mean_std[k]) / mean_std[6 + k];
        x[6] = x[7] = 0.f;
        // forward, layer by layer; lane l of a tile's result holds units
        // 4 (l / 16) + 0..3 of sample l % 16, and reads its operand columns back
        // as input 4 k + l / 16 of that sample
        if (slot == 0) {
#pragma unroll
            for (int k = 0; k < kMlpIn; k++) lds.col[kColX + k][j] = x[k];
            lds.col[kColOne][j] = 1.f;
        }
        const float x0 = slot == 0 ? x[0] : (slot == 1 ? x[1] : (slot == 2 ? x[2] : x[3]));
        const float x1 = slot == 0 ? x[4] : (slot == 1 ? x[5] : 0.f);
#pragma unroll
        for (int m = 0; m < 2; m++) {
            f32x4 d;
#pragma unroll
            for (int r = 0; r < 4; r++) d[r] = P[kOffB1 + 16 * m + 4 * slot + r];
            const float *w = P + kOffW1 + (16 * m + j) * kMlpIn;
            d = mfma_f32(w[slot], x0, d);
            d = mfma_f32(slot < 2 ? w[4 + (slot & 1)] : 0.f, x1, d);
#pragma unroll
            for (int r = 0; r < 4; r++) lds.col[kColH1 + 16 * m + 4 * slot + r][j] = lrelu(d[r]);
        }
    }
    __syncthreads();
    float h1[8], h2[8];
#pragma unroll
    for (int k = 0; k < 8; k++) h1[k] = lds.col[kColH1 + 4 * k + slot][j];
#pragma unroll
    for (int m = 0; m < 2; m++) {
        f32x4 d;
#pragma unroll
        for (int r = 0; r < 4; r++) d[r] = P[kOffB2 + 16 * m + 4 * slot + r];
#pragma unroll
        for (int k = 0; k < 8; k++) d = mfma_f32(P[kOffW2 + (16 * m + j) * kMlpH1 + 4 * k + slot], h1[k], d);
#pragma unroll
        for (int r = 0; r < 4; r++) lds.col[kColH2 + 16 * m + 4 * slot + r][j] = lrelu(d[r]);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 8; k++) h2[k] = lds.col[kColH2 + 4 * k + slot][j];
#pragma unroll
    for (int m = 0; m < 3; m++) {
        const bool row = 16 * m + j < kMlpOut;  // the last tile has four units
        f32x4 d;
#pragma unroll
        for (int r = 0; r < 4; r++) d[r] = 16 * m + 4 * slot + r < kMlpOut ? P[kOffB3 + 16 * m + 4 * slot + r] : 0.f;
#pragma unroll
        for (int k = 0; k < 8; k++)
            d = mfma_f32(row ? P[kOffW3 + (16 * m + j) * kMlpH2 + 4 * k + slot] : 0.f, h2[k], d);
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (16 * m + 4 * slot + r < kMlpOut) lds.col[kColDo + 16 * m + 4 * slot + r][j] = d[r];
    }
    __syncthreads();
    float L[36];
    {
        float o[kMlpOut];
#pragma unroll
        for (int k = 0; k < kMlpOut; k++) o[k] = lds.col[kColDo + k][j];
        cholesky_from_output(o, L);
    }
    // this slot's nine outputs: d loss / d o, summed over the draws in order
    constexpr int kPer = kMlpOut / 4;
    float dout[kPer], diag[kPer];
    int ia[kPer], ib[kPer];
#pragma unroll
    for (int e = 0; e < kPer; e++) {
        const int q = slot * kPer + e, ab = kCholIndex[q];
        ia[e] = ab >> 4;
        ib[e] = 8 + (ab & 15);
        dout[e] = 0.f;
        diag[e] = q < 8 ? __expf(lds.col[kColDo + q][j]) : 1.f;
    }
    const float bf = (float)(beta / 3.0);
    const float norm = 1.0f / ((float)batch * (float)draws);
    const M3<float> W = mul(U, A);
    float gW[8];
    project_algebra(W, gW);
    Stream rs(seed, (uint32_t)i, 0u, STREAM_TRAIN, step);
    double lacc = 0.0;
#pragma unroll 1
    for (int k0 = 0; k0 < draws; k0 += 4) {
        const int k = k0 + slot;
        float z[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, w[8], dw[8];
        if (zin) {
#pragma unroll
            for (int a = 0; a < 8; a++) z[a] = zin[((size_t)i * draws + (k < draws ? k : draws - 1)) * 8 + a];
        } else {
            // the stream gives every draw four outputs; this slot takes its own
#pragma unroll 1
            for (int t = 0; t < 4; t++) {
                float y[8];
#pragma unroll
                for (int a = 0; a < 8; a += 2) sym_draw_pair(rs, y[a], y[a + 1]);
#pragma unroll
                for (int a = 0; a < 8; a++) z[a] = t == slot ? y[a] : z[a];
            }
        }
        float w2 = 0.f;
#pragma unroll
        for (int a = 0; a < 8; a++) {
            float v = 0.f;
#pragma unroll
            for (int b = 0; b <= a; b++) v = fmaf(L[a * (a + 1) / 2 + b], z[b], v);
            w[a] = v;
            w2 = fmaf(v, v, w2);
        }
        const M3<float> Y = expand(algebra_from_omega<float>(w));
        const M3<float> YW = mul(Y, W);
        M3<float> Q = mul(W, Y);  // Q = YW + WY
        add_to(Q, YW);
        const float lin = retrace(YW);
        const float quad = retrace_mul(Y, YW);
        const float dS = -bf * (lin + 0.5f * quad);
        const float alpha = dS > 0.f ? __expf(-dS) : 1.f;
        if (valid && k < draws) lacc -= (double)(alpha * w2) * norm;
        float gQ[8];
        project_algebra(Q, gQ);
#pragma unroll
        for (int a = 0; a < 8; a++) {
            const float ddS = -bf * (gW[a] + 0.5f * gQ[a]);
            const float dalpha = dS > 0.f ? -alpha * ddS : 0.f;
            dw[a] = -(2.f * alpha * w[a] + w2 * dalpha) * norm;
        }
        __syncthreads();
#pragma unroll
        for (int a = 0; a < 8; a++) {
            lds.dz[slot][a][j] = dw[a];
            lds.dz[slot][8 + a][j] = z[a];
        }
        __syncthreads();
        const int nd = min(4, draws - k0);
        for (int t = 0; t < nd; t++) {
#pragma unroll
            for (int e = 0; e < kPer; e++) dout[e] = fmaf(lds.dz[t][ia[e]][j], lds.dz[t][ib[e]][j], dout[e]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kPer; e++) lds.col[kColDo + slot * kPer + e][j] = valid ? dout[e] * diag[e] : 0.f;
    __syncthreads();
    // backward: transposed weights, the slope of each unit from its activation's sign
    {
        float d9[9];
#pragma unroll
        for (int k = 0; k < 9; k++) d9[k] = lds.col[kColDo + 4 * k + slot][j];
#pragma unroll
        for (int m = 0; m < 2; m++) {
            f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < 9; k++) d = mfma_f32(P[kOffW3 + (4 * k + slot) * kMlpH2 + 16 * m + j], d9[k], d);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int u = 16 * m + 4 * slot + r;
                lds.col[kColDa2 + u][j] = lds.col[kColH2 + u][j] > 0.f ? d[r] : 0.01f * d[r];
            }
        }
    }
    __syncthreads();
    {
        float d8[8];
#pragma unroll
        for (int k = 0; k < 8; k++) d8[k] = lds.col[kColDa2 + 4 * k + slot][j];
#pragma unroll
        for (int m = 0; m < 2; m++) {
            f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < 8; k++) d = mfma_f32(P[kOffW2 + (4 * k + slot) * kMlpH1 + 16 * m + j], d8[k], d);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int u = 16 * m + 4 * slot + r;
                lds.col[kColDa1 + u][j] = lds.col[kColH1 + u][j] > 0.f ? d[r] : 0.01f * d[r];
            }
        }
    }
    __syncthreads();
    // the columns of these 16 samples, each as update_kernel's lanes read them:
    // entry 4 k + t holds sample 4 t + k
    float *out = inter + (size_t)blockIdx.x * kCols * kTrainSites;
#pragma unroll 4
    for (int c0 = 0; c0 < kCols; c0 += 4) {
        const int c = c0 + slot;
        if (c < kCols) out[c * kTrainSites + j] = lds.col[c][4 * (j & 3) + (j >> 2)];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) lacc += __shfl_down(lacc, off, 64);
    if (lane == 0) loss_partials[blockIdx.x] = lacc;
}

__device__ __forceinline__ unsigned short float_to_bf16(float v)
{
    const unsigned u = __float_as_uint(v);
    const unsigned r = u + 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even
    return (unsigned short)(r >> 16);
}

// The gradient of every parameter, sum over the batch of (derivative of a
// unit) x (input), FP64 products and sums in the samples' order, and with
// `adam` the Adam update.  One wavefront per block holds four 4 x 4 tiles of a
// layer's [units x (inputs, one)] matrix, the last column being the bias, as one
// v_mfma_f64_4x4x4 accumulator: each instruction adds four samples to 64
// parameters, one after the other with one rounding each (checked), so the
// sum is that of a plain loop over the batch.  The last block adds up the loss.
//
// What bounds it: the chain of batch / 4 dependent matrix instructions.  One
// thread per parameter looping over the batch (10 blocks, two uncoalesced
// loads an iteration) took 876 us at batch 4096, and Adam 5 us more; 19 us
// now.
constexpr int kTiles1 = 8 * 2, kTiles2 = 8 * 9, kTiles3 = 9 * 9, kTiles = kTiles1 + kTiles2 + kTiles3;
constexpr int kUpdateBlocks = (kTiles + 3) / 4;

__global__ __launch_bounds__(64) void update_kernel(const float *__restrict__ inter,
                                                    const double *__restrict__ loss_partials, int groups,
                                                    double *__restrict__ loss, float *__restrict__ grad, int adam,
                                                    float *__restrict__ params, float *__restrict__ m,
                                                    float *__restrict__ v, float lr, float c1, float c2,
                                                    unsigned short *__restrict__ bf16)
{
    const int lane = threadIdx.x;
    if (blockIdx.x == kUpdateBlocks) {
        double s = 0.0;
        for (int b = lane; b < groups; b += 64) s += loss_partials[b];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
        if (lane == 0) *loss = s;
        return;
    }
    // operands: lane l holds A[l % 4][l / 16] and B[l / 16][l % 4] of tile
    // (l / 4) % 4; result: row l / 16, column l % 4 of that tile
    const int tile = blockIdx.x * 4 + ((lane >> 2) & 3), unit = lane & 3, quad = lane >> 4;
    const bool live = tile < kTiles;
    const int t = live ? tile : kTiles - 1;
    int row, col, cols, ca, cb, offw, offb;
    if (t < kTiles1) {
        row = t >> 1, col = t & 1, cols = kMlpIn, ca = kColDa1, cb = kColX, offw = kOffW1, offb = kOffB1;
    } else if (t < kTiles1 + kTiles2) {
        row = (t - kTiles1) / 9, col = (t - kTiles1) % 9, cols = kMlpH1, ca = kColDa2, cb = kColH1, offw = kOffW2,
        offb = kOffB2;
    } else {
        row = (t - kTiles1 - kTiles2) / 9, col = (t - kTiles1 - kTiles2) % 9, cols = kMlpH2, ca = kColDo, cb = kColH2,
        offw = kOffW3, offb = kOffB3;
    }
    row *= 4, col *= 4;
    const int in = col + unit < cols ? cb + col + unit : kColOne;  // results beyond the bias column are not written
    // one buffer resource for a group's columns, moved on group by group
    constexpr int kStep = kCols * kTrainSites * (int)sizeof(float);
    const unsigned oa = ((ca + row + unit) * 4 + quad) * 16u, ob = (in * 4 + quad) * 16u;
    double s = 0.0;
    auto add_group = [&](const float4 &x, const float4 &y) {
        s = __builtin_amdgcn_mfma_f64_4x4x4f64((double)x.x, (double)y.x, s, 0, 0, 0);
        s = __builtin_amdgcn_mfma_f64_4x4x4f64((double)x.y, (double)y.y, s, 0, 0, 0);
        s = __builtin_amdgcn_mfma_f64_4x4x4f64((double)x.z, (double)y.z, s, 0, 0, 0);
        s = __builtin_amdgcn_mfma_f64_4x4x4f64((double)x.w, (double)y.w, s, 0, 0, 0);
    };
    // two sets of registers: one set's groups are in flight while the other's are added
    constexpr int kSet = 8;
    float4 a[2][kSet], b[2][kSet];
    auto load_set = [&](int which, int g0) {
#pragma unroll
        for (int k = 0; k < kSet; k++) {
            const size_t g = min(g0 + k, groups - 1);
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
                (void *)(inter + g * kCols * kTrainSites), (short)0, kStep, kBufferFlags);
            a[which][k] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, oa, 0, 0));
            b[which][k] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, ob, 0, 0));
        }
    };
    load_set(0, 0);
    int g0 = 0;
    for (; g0 + 2 * kSet <= groups; g0 += 2 * kSet) {
        load_set(1, g0 + kSet);
#pragma unroll
        for (int k = 0; k < kSet; k++) add_group(a[0][k], b[0][k]);
        load_set(0, g0 + 2 * kSet);
#pragma unroll
        for (int k = 0; k < kSet; k++) add_group(a[1][k], b[1][k]);
    }
    load_set(1, g0 + kSet);
#pragma unroll
    for (int k = 0; k < kSet; k++)
        if (g0 + k < groups) add_group(a[0][k], b[0][k]);
#pragma unroll
    for (int k = 0; k < kSet; k++)
        if (g0 + kSet + k < groups) add_group(a[1][k], b[1][k]);
    const int r = row + quad, c = col + unit;
    if (!live || c > cols) return;
    const int p = c < cols ? offw + r * cols + c : offb + r;
    const float g = (float)s;
    grad[p] = g;
    if (!adam) return;
    const float mm = 0.9f * m[p] + 0.1f * g;
    const float vv = 0.999f * v[p] + 0.001f * g * g;
    m[p] = mm;
    v[p] = vv;
    const float upd = lr * (mm / c1) / (sqrtf(vv / c2) + 1e-8f);
    params[p] -= upd;
    bf16[p] = float_to_bf16(params[p]);
}

__global__ __launch_bounds__(kBlock) void to_bf16_kernel(const float *__restrict__ params,
                                                         unsigned short *__restrict__ bf16)
{
    const int p = blockIdx.x * kBlock + threadIdx.x;
    if (p < kNParam) bf16[p] = float_to_bf16(params[p]);
}

// ---- sampling with the learned proposal ----------------------------------------
// What bounds it: the vector ALU (7400 instructions a wavefront, at 32^4 nearly all
// the time) and, beside it, LDS.  Against outputs and weights in plain rows
// (a sixth of the time went to bank conflicts) and a parameter at a time into
// LDS before the staple's loads: 24^3x48 79.5 -> 76.5 us a sub-sweep, 32^4 102 ->
// 99, 32^3x8 43 -> 38.5.
// WAVES: FP32 wavefronts per SIMD.  Four fit 128 VGPRs and, with the network's
// output buffer at 32 floats per link, 38.7 KB of LDS per block.  Three are ahead
// where four would leave a last block or two alone on a CU, and behind once there
// are many rounds (microseconds per sub-sweep, compressed, three | four):
//     blocks per CU    4.0    4.5    5.0    6.0    8.0    12    16
//                     62.0   69.9   70.6   79.5   99.4   145   196
//                     62.2   71.7   73.2   81.5   99.3   142   190
template <class T, int R, int WAVES>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? WAVES : 1, sizeof(T) == 4 ? WAVES : 2)))
void metropolis_learned_kernel(typename vec2<T>::type *__restrict__ f, Geom g, int mu, int parity, MetroParams prm,
                               const unsigned short *__restrict__ wbf16, const float *__restrict__ mean_std,
                               unsigned long long *__restrict__ count)
{
    __shared__ __align__(16) MlpImage im;
    __shared__ __align__(16) float obuf[kBlock / 64][64 * kMlpObuf];
    mlp_image_fill(im, wbf16, threadIdx.x, kBlock);
    const int h_raw = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
    const bool valid = h_raw < g.vh;
    const int h = valid ? h_raw : g.vh - 1;  // idle lanes mirror a real link for the network GEMMs, store nothing
    int n = 0;
    {
        const int idx = parity_index(g, parity, h);
        const Site x = site_of(g, idx);
        const M3<T> a = staple<T, R>(f, g, x, mu);
        M3<T> u = load_link<T, R>(f, g, mu, idx);
        float fe[6], o[36], L[36];
        staple_features(a, prm.beta, fe);
        __syncthreads();  // the image is whole; its loads travelled beside the staple's
        const bool learned =
            mlp_forward_mfma(im, mean_std, mean_std + 6, fe, obuf[threadIdx.x >> 6], o);  // whole wavefront
        cholesky_from_output(o, L);
        Stream rs(prm.seed, (uint32_t)lex_of(g, x), (uint32_t)mu, STREAM_LEARNED, prm.sweep);
        const double bf = prm.beta / 3.0;
        const T eps = T(prm.eps);
        const T x0abs = sqrt(T(1) - eps * eps);
        T tra = retrace_mul(u, a);
        int accepted = 0;
#pragma unroll 1
        for (int hit = 0; hit < prm.n_hit; hit++) {
            M3<T> xm;
            if (learned) {
                float z[8], om[8];
#pragma unroll
                for (int k = 0; k < 8; k += 2) sym_draw_pair(rs, z[k], z[k + 1]);
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    float v = 0.f;
#pragma unroll
                    for (int b = 0; b <= k; b++) v = fmaf(L[k * (k + 1) / 2 + b], z[b], v);
                    om[k] = v;
                }
                xm = exp_su3_proposal(algebra_from_omega<T>(om));
            } else {
                xm = rst_proposal<T>(rs, x0abs, eps);
            }
            const M3<T> v = propose_link<T, R>(xm, u);
            const T trv = retrace_mul(v, a);
            const T ds = T(-bf) * (trv - tra);
            if (accept_prob(ds) > rs.open()) {
                u = v;
                tra = trv;
                accepted++;
            }
        }
        if (valid) {
            if (prm.reunit) {
                M3<double> d = convert<double>(u);
                if constexpr (R == 2)
                    reunitarize<2, true>(d);  // the store keeps rows 0 and 1 only
                else
                    reunitarize_keep_det_sign<sizeof(T) == 4>(d);  // det U = +1 or -1 kept
                u = convert<T>(d);
            }
            store_link<T, R>(f, g, mu, idx, u);
            n = accepted;
        }
    }
    add_count(count, blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6), n);
}

// The sampling kernels' matrix-core forward pass on n given feature rows (6
// floats each): 36 outputs per row into out, and whether the row's
// standardised features are in range into ok.  A check of the network the
// sweeps evaluate; idle lanes of the last block mirror row n - 1.
__global__ __launch_bounds__(kBlock) void proposal_eval_kernel(const float *__restrict__ feat, int n,
                                                               const unsigned short *__restrict__ wbf16,
                                                               const float *__restrict__ mean_std,
                                                               float *__restrict__ out, int *__restrict__ ok)
{
    __shared__ __align__(16) MlpImage im;
    __shared__ __align__(16) float obuf[kBlock / 64][64 * kMlpObuf];
    mlp_image_fill(im, wbf16, threadIdx.x, kBlock);
    __syncthreads();
    const int i_raw = blockIdx.x * kBlock + threadIdx.x;
    const int i = i_raw < n ? i_raw : n - 1;
    float fe[kMlpIn], o[kMlpOut];
#pragma unroll
    for (int k = 0; k < kMlpIn; k++) fe[k] = feat[(size_t)kMlpIn * i + k];
    const bool in = mlp_forward_mfma(im, mean_std, mean_std + kMlpIn, fe, obuf[threadIdx.x >> 6], o);
    if (i_raw < n) {
#pragma unroll
        for (int k = 0; k < kMlpOut; k++) out[(size_t)kMlpOut * i + k] = o[k];
        ok[i] = in ? 1 : 0;
    }
}

// ---- launchers -------------------------------------------------------------------
void launch_proposal_eval(const float *feat, int n, const unsigned short *wbf16, const float *mean_std, float *out,
                          int *ok, hipStream_t s)
{
    proposal_eval_kernel<<<(n + kBlock - 1) / kBlock, kBlock, 0, s>>>(feat, n, wbf16, mean_std, out, ok);
}

template <class T, int R>
void launch_collect(const void *f, const Geom &g, int mu, int parity, int stride, float *out, size_t cap, size_t base,
                    hipStream_t s)
{
    const int n = (g.vh + stride - 1) / stride;
    collect_kernel<T, R><<<(n + kBlock - 1) / kBlock, kBlock, 0, s>>>((const typename vec2<T>::type *)f, g, mu, parity,
                                                                   stride, (float4 *)out, cap, base);
}

int feature_moments_blocks(size_t n)
{
    return (int)std::min<size_t>(kMomentBlocks, (n + kBlock - 1) / kBlock);
}

void launch_feature_moments(const float *smp, size_t cap, size_t n, double beta, double *partials, float *mean_std,
                            hipStream_t s)
{
    const int nb = feature_moments_blocks(n);
    feature_moments_kernel<<<nb, kBlock, 0, s>>>((const float4 *)smp, cap, n, beta, partials);
    feature_moments_finish<<<1, kBlock, 0, s>>>(partials, nb, n, mean_std);
}

size_t train_inter_floats(int batch)
{
    return (size_t)((batch + kTrainSites - 1) / kTrainSites) * kTrainSites * kCols;
}
int train_groups(int batch) { return (batch + kTrainSites - 1) / kTrainSites; }

void launch_train_step(const float *smp, size_t cap, size_t n_samples, int batch, int draws, uint64_t seed,
                       uint64_t step, double beta, float *params, const float *mean_std, const float *zin,
                       float *inter, double *loss_partials, double *loss, float *grad, float *m, float *v, float lr,
                       int adam_t, unsigned short *bf16, hipStream_t s)
{
    const int groups = train_groups(batch);
    train_kernel<<<groups, 64, 0, s>>>((const float4 *)smp, cap, n_samples, batch, draws, seed, step, beta, params,
                                       mean_std, zin, inter, loss_partials);
    const float c1 = 1.f - powf(0.9f, (float)adam_t), c2 = 1.f - powf(0.999f, (float)adam_t);
    update_kernel<<<kUpdateBlocks + 1, 64, 0, s>>>(inter, loss_partials, groups, loss, grad, adam_t > 0, params, m, v,
                                                   lr, c1, c2, bf16);
}

void launch_to_bf16(const float *params, unsigned short *bf16, hipStream_t s)
{
    to_bf16_kernel<<<(kNParam + kBlock - 1) / kBlock, kBlock, 0, s>>>(params, bf16);
}

template <class T, int R>
void launch_metropolis_learned(void *f, const Geom &g, int mu, int parity, const MetroParams &p,
                               const unsigned short *wbf16, const float *mean_std, unsigned long long *count,
                               hipStream_t s)
{
    const unsigned blocks = (unsigned)((g.vh + kBlock - 1) / kBlock);
    auto *links = (typename vec2<T>::type *)f;
    if constexpr (sizeof(T) == 4) {
        if (blocks <= 6 * 256) {  // the table at metropolis_learned_kernel; 256 CUs
            metropolis_learned_kernel<T, R, 3>
                <<<blocks, kBlock, 0, s>>>(links, g, mu, parity, p, wbf16, mean_std, count);
            return;
        }
    }
    metropolis_learned_kernel<T, R, 4><<<blocks, kBlock, 0, s>>>(links, g, mu, parity, p, wbf16, mean_std, count);
}

template void launch_collect<float, 3>(const void *, const Geom &, int, int, int, float *, size_t, size_t, hipStream_t);
template void launch_collect<float, 2>(const void *, const Geom &, int, int, int, float *, size_t, size_t, hipStream_t);
template void launch_collect<double, 3>(const void *, const Geom &, int, int, int, float *, size_t, size_t, hipStream_t);
template void launch_metropolis_learned<float, 3>(void *, const Geom &, int, int, const MetroParams &,
                                               const unsigned short *, const float *, unsigned long long *,
                                               hipStream_t);
template void launch_metropolis_learned<float, 2>(void *, const Geom &, int, int, const MetroParams &,
                                               const unsigned short *, const float *, unsigned long long *,
                                               hipStream_t);
template void launch_metropolis_learned<double, 3>(void *, const Geom &, int, int, const MetroParams &,
                                                const unsigned short *, const float *, unsigned long long *,
                                                hipStream_t);

} // namespace glacx
