// mc_mlp.h - the warm-start network of the per-cell balance: a 72 -> 128 ->
// 128 -> 128 -> 31 ReLU perceptron, BF16 weights and activations, FP32
// accumulation on the matrix cores (v_mfma_f32_16x16x32_bf16), trained on
// the device by its own forward, backward and Adam kernels.
//
// Features of a cell (72): log10 of J summed over 64 contiguous groups of
// frequency bins, log10 nH, log10 of the abundances of H, He, C, N, O, Ne, S.
// Targets (31): log10 Te and log10 of the ionic fractions of those seven
// elements, stages 1..min(Z+1, 5) (2 + 3 + 5*5 = 30).  Both are standardised
// with per-column mean and standard deviation held with the network.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mcm {

constexpr int kBands = 64;
constexpr int kIn = 72, kInP = 96;       // inputs, padded to a multiple of 32
constexpr int kHid = 128;
constexpr int kOut = 31, kOutP = 32;
constexpr int kLayers = 4;
constexpr int kSlotsZ[7] = { 1, 2, 6, 7, 8, 10, 16 };
constexpr int kStageMax = 5;

__host__ __device__ constexpr int layer_in(int l) { return l == 0 ? kInP : kHid; }
__host__ __device__ constexpr int layer_out(int l) { return l == kLayers - 1 ? kOutP : kHid; }
// flat FP32 parameter vector: W_l [out][in] then b_l [out], layer after layer
__host__ __device__ constexpr int w_off(int l)
{
    return l == 0 ? 0 : w_off(l - 1) + layer_out(l - 1) * layer_in(l - 1) + layer_out(l - 1);
}
__host__ __device__ constexpr int b_off(int l) { return w_off(l) + layer_out(l) * layer_in(l); }
constexpr int kParams = w_off(kLayers);  // 49,568
constexpr int kWeightsBf16 = kParams;     // bf16 copies of W (the b slots unused)

struct Net {
    const uint16_t *W;    // bf16 copy of the parameters (W_l at w_off(l), [out][in])
    const float *P;       // fp32 master parameters (biases read from here)
};

// column scaling of features and targets: x_std = (x - mean) / std
struct Scale {
    const float *xmean, *xstd, *ymean, *ystd;
};

// What a training step keeps of a batch: BF16 inputs, hidden activations and
// back-propagated rows as [tile][feature][16 rows]; layer l of H and D at
// l * stride.
struct TrainBuf {
    uint16_t *X, *H, *D, *D3;
    size_t stride;
};

}  // namespace mcm

// launchers (mc_mlp.hip); every pointer is device memory.
// forward: X0 bf16 [n][kInP] -> Y fp32 [n][ldy] (standardised outputs)
hipError_t mcm_forward(const uint16_t *X0, int n, mcm::Net net, float *Y, int ldy, int blocks, hipStream_t s);
// A batch of n rows: an even number of 16-row tiles (zero rows fill the
// last), and the slices its gradient is formed in (at least 8 steps of 32
// rows each, 16 slices at most: 4096 rows and more fill the chip).
inline int mcm_train_tiles(int n) { return (n + 31) / 32 * 2; }
inline int mcm_train_slices(int n)
{
    const int s = mcm_train_tiles(n) / 16;
    return s < 1 ? 1 : s > 16 ? 16 : s;
}
// its working memory in BF16 elements
inline size_t mcm_train_elems(int n)
{
    return (size_t)mcm_train_tiles(n) * 16 * (mcm::kInP + 6 * mcm::kHid + mcm::kOutP);
}
// W (published BF16) transposed per layer: [in][out] at w_off
hipError_t mcm_transpose(const uint16_t *W, uint16_t *WT, hipStream_t s);
// gradient of L = sum M (Y - T)^2 over rows idx[0..n) of a raw data set:
// part [mcm_train_slices(n)][kParams] gets the slices of the unnormalised
// gradient 2 sum M (Y - T) dY/dP; sums[0] += sum M (Y-T)^2, sums[1] += sum M
// (zero them first).  mem: mcm_train_elems(n).
hipError_t mcm_gradient(const float *Xs, const float *Ts, const float *Ms, const int *idx, int n, mcm::Scale sc,
                        mcm::Net net, const uint16_t *WT, uint16_t *mem, float *part, double *sums, int blocks,
                        hipStream_t s);
hipError_t mcm_sum(const float *part, int slices, float *grad, hipStream_t s);
// Adam step t (1-based) on the sum of the slices / sums[1]; refreshes the
// BF16 copies
hipError_t mcm_adam(float *P, const float *part, int slices, float *m, float *v, const double *sums, int t,
                    float lr, uint16_t *W, uint16_t *WT, hipStream_t s);
// first entry of X (bad[0]) and of T or M (bad[1]) that is not finite, or
// negative in M; all ones where there is none
hipError_t mcm_check(const float *X, size_t nx, const float *T, const float *M, size_t nt, unsigned long long *bad,
                     hipStream_t s);
hipError_t mcm_publish(const float *P, uint16_t *W, hipStream_t s);
hipError_t mcm_standardise(const float *Xraw, int n, mcm::Scale sc, uint16_t *X0, hipStream_t s);
hipError_t mcm_unscale(float *Y, int n, int ldy, mcm::Scale sc, hipStream_t s);
