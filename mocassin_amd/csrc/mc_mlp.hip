// mc_mlp.hip - kernels of the warm-start network (see mc_mlp.h): the fused
// forward pass, the training step, and the data movers around them.
//
// Matrix products use v_mfma_f32_16x16x32_bf16 (one 64-lane wavefront
// computes a 16x16 FP32 tile from 16x32 and 32x16 BF16 operands).  Operand
// layout of that instruction: lane l supplies A[l%16][(l/16)*8 + 0..7] and
// B[(l/16)*8 + 0..7][l%16] and receives D[(l/16)*4 + 0..3][l%16].
#include "mc_mlp.h"

namespace mcm {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// round to nearest even (operands are finite)
__device__ __forceinline__ uint16_t f2bf(float f)
{
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ __forceinline__ bf16x8 ld8(const uint16_t *p)
{
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(p));
}

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// w_off and b_off of a layer known at run time only
__device__ __forceinline__ int w_at(int l)
{
    constexpr int o[kLayers + 1] = { w_off(0), w_off(1), w_off(2), w_off(3), kParams };
    return l == 0 ? o[0] : l == 1 ? o[1] : l == 2 ? o[2] : l == 3 ? o[3] : o[4];
}
__device__ __forceinline__ int b_at(int l) { return w_at(l) + layer_out(l) * layer_in(l); }

// ------------------------------------------------------------- forward
// LDS: the four weight matrices (row stride in + 8 to spread banks), the
// biases, and per wavefront two 16-row activation buffers (stride 136).
constexpr int kActS = kHid + 8;
constexpr int kTile = 64;                       // rows per workgroup tile (4 wavefronts x 16)
__host__ __device__ constexpr int lw_stride(int l) { return layer_in(l) + 8; }
__host__ __device__ constexpr int lw_off(int l)
{
    return l == 0 ? 0 : lw_off(l - 1) + layer_out(l - 1) * lw_stride(l - 1);
}
__device__ __forceinline__ int lw_at(int l)
{
    constexpr int o[kLayers] = { lw_off(0), lw_off(1), lw_off(2), lw_off(3) };
    return l == 0 ? o[0] : l == 1 ? o[1] : l == 2 ? o[2] : o[3];
}
constexpr int kLdsW = lw_off(kLayers);                                   // bf16 elements
constexpr int kLdsBias = kHid * 3 + kOutP;                               // floats
constexpr int kLdsAct = 4 * 2 * 16 * kActS;                              // bf16 elements
constexpr size_t kFwdLds = (size_t)kLdsW * 2 + (size_t)kLdsBias * 4 + (size_t)kLdsAct * 2;

__global__ void __launch_bounds__(256) forward_kernel(const uint16_t *__restrict__ X0, int n, Net net,
                                                      float *__restrict__ Y, int ldy)
{
    extern __shared__ __align__(16) unsigned char lds[];
    uint16_t *Ws = reinterpret_cast<uint16_t *>(lds);
    float *bias = reinterpret_cast<float *>(lds + (size_t)kLdsW * 2);
    uint16_t *act = reinterpret_cast<uint16_t *>(lds + (size_t)kLdsW * 2 + (size_t)kLdsBias * 4);
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    // weights and biases into LDS, 16 bytes at a time
    for (int l = 0; l < kLayers; ++l) {
        const int K = layer_in(l), N = layer_out(l), vpr = K / 8;
        const uint16_t *src = net.W + w_at(l);
        for (int e = tid; e < N * vpr; e += 256) {
            const int r = e / vpr, v = e % vpr;
            *reinterpret_cast<uint4 *>(Ws + lw_at(l) + r * lw_stride(l) + v * 8) =
                *reinterpret_cast<const uint4 *>(src + (size_t)r * K + v * 8);
        }
    }
    for (int e = tid; e < kLdsBias; e += 256) {
        const int l = e < 3 * kHid ? e / kHid : 3, j = e < 3 * kHid ? e % kHid : e - 3 * kHid;
        bias[e] = net.P[b_at(l) + j];
    }
    uint16_t *a0 = act + (size_t)(w * 2) * 16 * kActS, *a1 = a0 + 16 * kActS;
    const int ntiles = (n + kTile - 1) / kTile;
    const int lr = lane & 15, lk = (lane >> 4) * 8, lrow = (lane >> 4) * 4;
    __syncthreads();
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int r0 = tile * kTile + w * 16;
        for (int e = lane; e < 16 * (kInP / 8); e += 64) {
            const int r = e / (kInP / 8), v = e % (kInP / 8);
            uint4 val = make_uint4(0, 0, 0, 0);
            if (r0 + r < n) val = *reinterpret_cast<const uint4 *>(X0 + (size_t)(r0 + r) * kInP + v * 8);
            *reinterpret_cast<uint4 *>(a0 + r * kActS + v * 8) = val;
        }
        __syncthreads();
        for (int l = 0; l < kLayers; ++l) {
            const uint16_t *in = (l & 1) ? a1 : a0;
            uint16_t *out = (l & 1) ? a0 : a1;
            const int K = layer_in(l), N = layer_out(l);
            const uint16_t *Wl = Ws + lw_at(l);
            const float *bl = bias + l * kHid;
            for (int t = 0; t < N / 16; ++t) {
                f32x4 acc = { 0.f, 0.f, 0.f, 0.f };
                for (int s = 0; s < K / 32; ++s) {
                    const bf16x8 a = ld8(in + lr * kActS + 32 * s + lk);
                    const bf16x8 b = ld8(Wl + (16 * t + lr) * lw_stride(l) + 32 * s + lk);
                    acc = mfma(a, b, acc);
                }
                const int col = 16 * t + lr;
                for (int i = 0; i < 4; ++i) {
                    const int row = lrow + i;
                    float v = acc[i] + bl[col];
                    if (l < kLayers - 1) {
                        v = v > 0.f ? v : 0.f;
                        out[row * kActS + col] = f2bf(v);
                    } else if (col < kOut && r0 + row < n) {
                        Y[(size_t)(r0 + row) * ldy + col] = v;
                    }
                }
            }
            __syncthreads();
        }
    }
}

__device__ __forceinline__ float stdz(float x, float mean, float sd) { return (x - mean) / sd; }

template <int S> struct Steps { static constexpr int value = S; };

// ------------------------------------------------------------- training
// A training step is three launches: step_kernel takes 16 rows at a time
// through standardisation, forward pass, loss and backward pass; grad_kernel
// forms the weight and bias gradients of slices of the batch; adam_kernel
// adds the slices in order and updates.  The rounding points are those of
// the layers one by one: BF16 inputs, activations and back-propagated rows,
// FP32 sums on the matrix cores.
//
// The step is bound by latency (a 4096-row batch is 4 GFLOP): so a workgroup
// loads every weight fragment it will use into registers at its start, 44 of
// them a lane, all in flight at once, and then needs nothing but LDS between
// its layers.  Inputs, activations and back-propagated rows go to memory as
// [tile][feature][16 rows]: a lane's four rows of a result are 8 contiguous
// bytes, and grad_kernel, whose inner index is the row, reads its fragments
// 16 bytes a lane without staging.  One step of 4096 rows: 181 us of
// kernels as 14 launches of one operation each, 28 now (18 + 6 + 4).
constexpr int kRows = 16;                      // rows of a tile
constexpr int kTrainS = kHid + 8;              // LDS row stride of a tile

// the four wavefronts of a workgroup share a tile; wavefront w computes the
// feature tiles 2 w and 2 w + 1 of a layer
__global__ void __launch_bounds__(256, 1) step_kernel(const float *__restrict__ Xs, const float *__restrict__ Ts,
                                                      const float *__restrict__ Ms, const int *__restrict__ idx,
                                                      int n, int tiles, Scale sc, Net net,
                                                      const uint16_t *__restrict__ WT, TrainBuf B,
                                                      double *__restrict__ sums)
{
    __shared__ __align__(16) uint16_t buf[2][kRows * kTrainS];
    __shared__ float bias[3 * kHid + kOutP], xs[2 * kIn], ys[2 * kOut];
    __shared__ double red[2][4];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int lr = lane & 15, lk = (lane >> 4) * 8, lrow = (lane >> 4) * 4;
    // A tile's rows of the data set, all loads of a kind in flight together:
    // inputs, then targets and masks of the outputs this lane will see (w <
    // 2); rows beyond the batch and padded columns load in range.  The data
    // of the tile after, and the row numbers of the one after that, are on
    // their way while a tile is worked on.
    constexpr int kE = kRows * kInP / 256;
    const int oc = 16 * w + lr;
    int row[kE], orow[4];
    float xn[kE], tn[4], mn[4];
    auto load_rows = [&](int tile) {
        const int r0 = min(tile, tiles) * kRows;
#pragma unroll
        for (int u = 0; u < kE; ++u) row[u] = idx[min(n - 1, r0 + (tid + 256 * u) / kInP)];
#pragma unroll
        for (int i = 0; i < 4; ++i) orow[i] = idx[min(n - 1, r0 + lrow + i)];
    };
    auto load_data = [&] {
#pragma unroll
        for (int u = 0; u < kE; ++u) xn[u] = Xs[(size_t)row[u] * kIn + min(kIn - 1, (tid + 256 * u) % kInP)];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const size_t src = (size_t)orow[i] * kOut + min(kOut - 1, oc);
            tn[i] = Ts[src];
            mn[i] = Ms[src];
        }
    };
    load_rows(blockIdx.x);
    for (int e = tid; e < 2 * kIn; e += 256) xs[e] = e < kIn ? sc.xmean[e] : sc.xstd[e - kIn];
    for (int e = tid; e < 2 * kOut; e += 256) ys[e] = e < kOut ? sc.ymean[e] : sc.ystd[e - kOut];
    load_data();
    load_rows(blockIdx.x + gridDim.x);
    // forward fragments W_l[out 16 t + lr][in 32 s + lk ..], backward
    // WT_l[in 16 t + lr][out 32 s + lk ..]
    constexpr int w0 = w_off(0), w1 = w_off(1), w2 = w_off(2), w3 = w_off(3);
    bf16x8 f0[2][3], f1[2][4], f2[2][4], f3[4], b3[2], b2[2][4], b1[2][4];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int o = 16 * (2 * w + u) + lr;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if (s < 3) f0[u][s] = ld8(net.W + w0 + o * kInP + 32 * s + lk);
            f1[u][s] = ld8(net.W + w1 + o * kHid + 32 * s + lk);
            f2[u][s] = ld8(net.W + w2 + o * kHid + 32 * s + lk);
            b2[u][s] = ld8(WT + w2 + o * kHid + 32 * s + lk);
            b1[u][s] = ld8(WT + w1 + o * kHid + 32 * s + lk);
        }
        b3[u] = ld8(WT + w3 + o * kOutP + lk);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) f3[s] = ld8(net.W + w3 + (16 * (w & 1) + lr) * kHid + 32 * s + lk);
    for (int e = tid; e < 3 * kHid + kOutP; e += 256) {
        const int l = e < 3 * kHid ? e / kHid : 3;
        bias[e] = net.P[b_at(l) + e - l * kHid];
    }
    double l2 = 0.0, mm = 0.0;
    __syncthreads();

    for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const int r0 = tile * kRows;
        float xv[kE], tv[4], mv[4];
#pragma unroll
        for (int u = 0; u < kE; ++u) xv[u] = xn[u];
#pragma unroll
        for (int i = 0; i < 4; ++i) { tv[i] = tn[i]; mv[i] = mn[i]; }
        if (tile + (int)gridDim.x < tiles) {
            load_data();
            load_rows(tile + 2 * (int)gridDim.x);
        }
#pragma unroll
        for (int u = 0; u < kE; ++u) {
            const int r = (tid + 256 * u) / kInP, j = (tid + 256 * u) % kInP, k = min(kIn - 1, j);
            const uint16_t v = f2bf(stdz(xv[u], xs[k], xs[kIn + k]));
            buf[0][r * kTrainS + j] = j < kIn && r0 + r < n ? v : (uint16_t)0;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = min(kOut - 1, oc);
            const bool on = oc < kOut && r0 + lrow + i < n;
            tv[i] = on ? stdz(tv[i], ys[k], ys[kOut + k]) : 0.f;
            mv[i] = on ? mv[i] : 0.f;
        }
        __syncthreads();
        if (tid < 2 * kInP) {
            uint16_t q[8];
            for (int i = 0; i < 8; ++i) q[i] = buf[0][((tid & 1) * 8 + i) * kTrainS + tid / 2];
            *reinterpret_cast<uint4 *>(B.X + ((size_t)tile * kInP + tid / 2) * kRows + (tid & 1) * 8) =
                __builtin_bit_cast(uint4, q);
        }
        unsigned on[3] = { 0u, 0u, 0u };        // a bit per hidden activation above zero
        // one layer: `in` times the fragments, through `store` per feature
        auto product = [&](const uint16_t *in, auto steps, auto frag, auto store) {
            constexpr int S = decltype(steps)::value;
            bf16x8 a[S];
#pragma unroll
            for (int s = 0; s < S; ++s) a[s] = ld8(in + lr * kTrainS + 32 * s + lk);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                f32x4 acc = { 0.f, 0.f, 0.f, 0.f };
#pragma unroll
                for (int s = 0; s < S; ++s) acc = mfma(a[s], frag(u, s), acc);
                store(u, 16 * (2 * w + u) + lr, acc);
            }
        };
        // four rows of a feature to LDS and to memory
        auto put = [&](uint16_t *out, uint16_t *mem, int col, const uint16_t *q) {
            if (out)
#pragma unroll
                for (int i = 0; i < 4; ++i) out[(lrow + i) * kTrainS + col] = q[i];
            *reinterpret_cast<uint2 *>(mem + ((size_t)tile * kHid + col) * kRows + lrow) =
                make_uint2(q[0] | (unsigned)q[1] << 16, q[2] | (unsigned)q[3] << 16);
        };
        auto hidden = [&](int l, uint16_t *out) {
            return [&, l, out](int u, int col, const f32x4 &acc) {
                uint16_t q[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float v = acc[i] + bias[l * kHid + col];
                    q[i] = f2bf(v > 0.f ? v : 0.f);
                    if (q[i]) on[l] |= 1u << (4 * u + i);
                }
                put(out, B.H + (size_t)l * B.stride, col, q);
            };
        };
        auto back = [&](int l, uint16_t *out) {
            return [&, l, out](int u, int col, const f32x4 &acc) {
                uint16_t q[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) q[i] = f2bf(on[l] >> (4 * u + i) & 1u ? acc[i] : 0.f);
                put(out, B.D + (size_t)l * B.stride, col, q);
            };
        };
        product(buf[0], Steps<3>{}, [&](int u, int s) { return f0[u][s]; }, hidden(0, buf[1]));
        __syncthreads();
        product(buf[1], Steps<4>{}, [&](int u, int s) { return f1[u][s]; }, hidden(1, buf[0]));
        __syncthreads();
        product(buf[0], Steps<4>{}, [&](int u, int s) { return f2[u][s]; }, hidden(2, buf[1]));
        __syncthreads();
        // outputs and dY = 2 M (Y - T): feature tile w of two
        if (w < 2) {
            f32x4 acc = { 0.f, 0.f, 0.f, 0.f };
#pragma unroll
            for (int s = 0; s < 4; ++s) acc = mfma(ld8(buf[1] + lr * kTrainS + 32 * s + lk), f3[s], acc);
            uint16_t q[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float d = acc[i] + bias[3 * kHid + oc] - tv[i], m = mv[i];
                q[i] = f2bf(oc < kOut && r0 + lrow + i < n ? 2.f * m * d : 0.f);
                l2 += (double)m * (double)d * (double)d;
                mm += (double)m;
                buf[0][(lrow + i) * kTrainS + oc] = q[i];
            }
            *reinterpret_cast<uint2 *>(B.D3 + ((size_t)tile * kOutP + oc) * kRows + lrow) =
                make_uint2(q[0] | (unsigned)q[1] << 16, q[2] | (unsigned)q[3] << 16);
        }
        __syncthreads();
        product(buf[0], Steps<1>{}, [&](int u, int) { return b3[u]; }, back(2, buf[1]));
        __syncthreads();
        product(buf[1], Steps<4>{}, [&](int u, int s) { return b2[u][s]; }, back(1, buf[0]));
        __syncthreads();
        product(buf[0], Steps<4>{}, [&](int u, int s) { return b1[u][s]; }, back(0, nullptr));
        __syncthreads();
    }
    for (int o = 32; o >= 1; o >>= 1) {
        l2 += __shfl_xor(l2, o);
        mm += __shfl_xor(mm, o);
    }
    if (lane == 0) { red[0][w] = l2; red[1][w] = mm; }
    __syncthreads();
    if (tid < 2) atomicAdd(&sums[tid], red[tid][0] + red[tid][1]);      // wavefronts 2 and 3 see no output
}

// dW_l[out][in] = sum over rows of dZ_l[out] prev_l[in], db_l = sum of dZ_l:
// one wavefront per 32 x 32 weights and slice of `per` steps of 32 rows,
// into part[slice][parameter].
constexpr int kGradTiles = 4 * 3 + 4 * 4 + 4 * 4 + 1 * 4;
__global__ void __launch_bounds__(64) grad_kernel(TrainBuf B, int steps, int per, float *__restrict__ part)
{
    const int lane = threadIdx.x, g = lane >> 4, lr = lane & 15, lrow = g * 4;
    int t = blockIdx.x, l = 0;
    if (t >= 12) { t -= 12; l = 1; }
    if (l == 1 && t >= 16) { t -= 16; l = 2; }
    if (l == 2 && t >= 16) { t -= 16; l = 3; }
    const int nd = l == 3 ? kOutP : kHid, np = l == 0 ? kInP : kHid;
    const int n0 = t / (np / 32) * 32, k0 = t % (np / 32) * 32;
    // rows 8 g .. of 32: tile g / 2 of two, half g % 2
    const uint16_t *dz = (l == 3 ? B.D3 : B.D + (size_t)l * B.stride) + ((size_t)(g >> 1) * nd + n0 + lr) * kRows + (g & 1) * 8;
    const uint16_t *pv = (l == 0 ? B.X : B.H + (size_t)(l - 1) * B.stride) + ((size_t)(g >> 1) * np + k0 + lr) * kRows + (g & 1) * 8;
    f32x4 acc[2][2];
    float db[2] = { 0.f, 0.f };
    for (int a = 0; a < 2; ++a)
        for (int b = 0; b < 2; ++b) acc[a][b] = f32x4{ 0.f, 0.f, 0.f, 0.f };
    const int s0 = blockIdx.y * per, s1 = min(steps, s0 + per);
    // `U` steps with their loads in flight together
    auto sum = [&](int s, auto unroll) {
        constexpr int U = decltype(unroll)::value;
        bf16x8 A[U][2], P[U][2];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                A[u][a] = ld8(dz + ((size_t)(s + u) * 2 * nd + 16 * a) * kRows);
                P[u][a] = ld8(pv + ((size_t)(s + u) * 2 * np + 16 * a) * kRows);
            }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int a = 0; a < 2; ++a) {
#pragma unroll
                for (int b = 0; b < 2; ++b) acc[a][b] = mfma(A[u][a], P[u][b], acc[a][b]);
#pragma unroll
                for (int i = 0; i < 8; ++i) db[a] += (float)A[u][a][i];
            }
    };
    int s = s0;
    for (; s + 8 <= s1; s += 8) sum(s, Steps<8>{});
    for (; s < s1; ++s) sum(s, Steps<1>{});
    float *out = part + (size_t)blockIdx.y * kParams;
    for (int a = 0; a < 2; ++a) {
        for (int b = 0; b < 2; ++b)
            for (int i = 0; i < 4; ++i)
                out[w_at(l) + (n0 + 16 * a + lrow + i) * np + k0 + 16 * b + lr] = acc[a][b][i];
        if (k0 == 0) {
            db[a] += __shfl_xor(db[a], 16);
            db[a] += __shfl_xor(db[a], 32);
            if (g == 0) out[b_at(l) + n0 + 16 * a + lr] = db[a];
        }
    }
}

__device__ __forceinline__ float slice_sum(const float *part, int slices, int i)
{
    float g = 0.f;
#pragma unroll 8
    for (int s = 0; s < slices; ++s) g += part[(size_t)s * kParams + i];
    return g;
}

__global__ void sum_kernel(const float *__restrict__ part, int slices, float *__restrict__ grad)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kParams) grad[i] = slice_sum(part, slices, i);
}

// where the transposed copy holds parameter i (biases: -1)
__device__ __forceinline__ int transposed(int i)
{
    int l = 0;
    while (l < kLayers - 1 && i >= w_at(l + 1)) ++l;
    const int e = i - w_at(l), K = layer_in(l), N = layer_out(l);
    return e < N * K ? w_at(l) + e % K * N + e / K : -1;
}

__global__ void transpose_kernel(const uint16_t *__restrict__ W, uint16_t *__restrict__ WT)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= kParams) return;
    const int t = transposed(i);
    if (t >= 0) WT[t] = W[i];
}

__global__ void adam_kernel(float *__restrict__ P, const float *__restrict__ part, int slices, float *__restrict__ m,
                            float *__restrict__ v, const double *__restrict__ sums, float c1, float c2,
                            float lr, uint16_t *__restrict__ W, uint16_t *__restrict__ WT)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= kParams) return;
    const float scale = sums[1] > 0.0 ? (float)(1.0 / sums[1]) : 0.f;
    const float g = slice_sum(part, slices, i) * scale;
    const float mi = 0.9f * m[i] + 0.1f * g;
    const float vi = 0.999f * v[i] + 0.001f * g * g;
    m[i] = mi;
    v[i] = vi;
    const float p = P[i] - lr * (mi / c1) / (sqrtf(vi / c2) + 1e-8f);
    P[i] = p;
    W[i] = f2bf(p);
    const int t = transposed(i);
    if (t >= 0) WT[t] = f2bf(p);
}

__global__ void __launch_bounds__(256) check_kernel(const float *__restrict__ X, size_t nx, const float *__restrict__ T,
                                                    const float *__restrict__ M, size_t nt,
                                                    unsigned long long *__restrict__ bad)
{
    const size_t step = (size_t)gridDim.x * blockDim.x, i0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    unsigned long long x = ~0ull, t = ~0ull;
    for (size_t i = i0; i < nx; i += step)
        if (!isfinite(X[i])) { x = i; break; }
    for (size_t i = i0; i < nt; i += step)
        if (!isfinite(T[i]) || !isfinite(M[i]) || M[i] < 0.f) { t = i; break; }
    if (x != ~0ull) atomicMin(&bad[0], x);
    if (t != ~0ull) atomicMin(&bad[1], t);
}

__global__ void publish_kernel(const float *__restrict__ P, uint16_t *__restrict__ W)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kParams) W[i] = f2bf(P[i]);
}

__global__ void standardise_kernel(const float *__restrict__ X, int n, Scale sc, uint16_t *__restrict__ X0)
{
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (long)n * kInP) return;
    const long r = e / kInP;
    const int j = (int)(e % kInP);
    X0[e] = j < kIn ? f2bf(stdz(X[r * kIn + j], sc.xmean[j], sc.xstd[j])) : (uint16_t)0;
}

__global__ void unscale_kernel(float *__restrict__ Y, int n, int ldy, Scale sc)
{
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (long)n * kOut) return;
    const long r = e / kOut;
    const int j = (int)(e % kOut);
    Y[r * ldy + j] = Y[r * ldy + j] * sc.ystd[j] + sc.ymean[j];
}

}  // namespace mcm

using namespace mcm;

static unsigned grid1(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

hipError_t mcm_forward(const uint16_t *X0, int n, Net net, float *Y, int ldy, int blocks, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    static bool attr = false;
    if (!attr) {
        hipError_t e = hipFuncSetAttribute((const void *)forward_kernel,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)kFwdLds);
        if (e != hipSuccess) return e;
        attr = true;
    }
    const int ntiles = (n + kTile - 1) / kTile;
    const int g = ntiles < blocks ? ntiles : blocks;
    hipLaunchKernelGGL(forward_kernel, dim3(g), dim3(256), kFwdLds, s, X0, n, net, Y, ldy);
    return hipGetLastError();
}

TrainBuf mcm_train_buf(uint16_t *mem, int n)
{
    const int t = mcm_train_tiles(n);
    TrainBuf B;
    B.stride = (size_t)t * kHid * kRows;
    B.X = mem;
    B.H = B.X + (size_t)t * kInP * kRows;
    B.D = B.H + 3 * B.stride;
    B.D3 = B.D + 3 * B.stride;
    return B;
}

hipError_t mcm_transpose(const uint16_t *W, uint16_t *WT, hipStream_t s)
{
    hipLaunchKernelGGL(transpose_kernel, dim3(grid1(kParams, 256)), dim3(256), 0, s, W, WT);
    return hipGetLastError();
}

hipError_t mcm_gradient(const float *Xs, const float *Ts, const float *Ms, const int *idx, int n, Scale sc, Net net,
                        const uint16_t *WT, uint16_t *mem, float *part, double *sums, int blocks, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    const TrainBuf B = mcm_train_buf(mem, n);
    const int tiles = mcm_train_tiles(n), steps = tiles / 2, slices = mcm_train_slices(n);
    hipLaunchKernelGGL(step_kernel, dim3(tiles < blocks ? tiles : blocks), dim3(256), 0, s, Xs, Ts, Ms, idx, n, tiles,
                       sc, net, WT, B, sums);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(grad_kernel, dim3(kGradTiles, slices), dim3(64), 0, s, B, steps, (steps + slices - 1) / slices,
                       part);
    return hipGetLastError();
}

hipError_t mcm_sum(const float *part, int slices, float *grad, hipStream_t s)
{
    hipLaunchKernelGGL(sum_kernel, dim3(grid1(kParams, 256)), dim3(256), 0, s, part, slices, grad);
    return hipGetLastError();
}

hipError_t mcm_adam(float *P, const float *part, int slices, float *m, float *v, const double *sums, int t, float lr,
                    uint16_t *W, uint16_t *WT, hipStream_t s)
{
    const float c1 = 1.f - powf(0.9f, (float)t), c2 = 1.f - powf(0.999f, (float)t);
    hipLaunchKernelGGL(adam_kernel, dim3(grid1(kParams, 256)), dim3(256), 0, s, P, part, slices, m, v, sums, c1, c2, lr,
                       W, WT);
    return hipGetLastError();
}

hipError_t mcm_check(const float *X, size_t nx, const float *T, const float *M, size_t nt, unsigned long long *bad,
                     hipStream_t s)
{
    hipError_t e = hipMemsetAsync(bad, 0xff, 2 * sizeof(unsigned long long), s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(check_kernel, dim3(2048), dim3(256), 0, s, X, nx, T, M, nt, bad);
    return hipGetLastError();
}

hipError_t mcm_publish(const float *P, uint16_t *W, hipStream_t s)
{
    hipLaunchKernelGGL(publish_kernel, dim3(grid1(kParams, 256)), dim3(256), 0, s, P, W);
    return hipGetLastError();
}

hipError_t mcm_standardise(const float *Xraw, int n, Scale sc, uint16_t *X0, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(standardise_kernel, dim3(grid1((long)n * kInP, 256)), dim3(256), 0, s, Xraw, n, sc, X0);
    return hipGetLastError();
}

hipError_t mcm_unscale(float *Y, int n, int ldy, Scale sc, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(unscale_kernel, dim3(grid1((long)n * kOut, 256)), dim3(256), 0, s, Y, n, ldy, sc);
    return hipGetLastError();
}
