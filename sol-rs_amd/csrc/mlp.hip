// mlp.hip -- the radiance cache's network: a 64-input MLP with four hidden
// ReLU layers of width 64 and 3 linear outputs, no biases, BF16 operands on
// MFMA (v_mfma_f32_16x16x32_bf16) with FP32 accumulation, trained by
// hand-written backward kernels and Adam with FP32 master weights.
//
// Parameters (FP32 master, P = 4*64*64 + 64*16 = 17408 floats):
//   W_l[k][n] at l*4096 + k*64 + n        (l = 0..3, k = input, n = output)
//   W_4[k][n] at 16384 + k*16 + n         (n < 3 used; columns 3..15 stay 0)
// BF16 copies: "forward" layout Wt_l[n][k] (operand B of X*W with k
// contiguous) and "backward" layout = the master layout (operand B of dY*W^T).
//
// MFMA 16x16x32 lane layout (lane l, r = l % 16, q = l / 16):
//   A (16 x 32): row r, k = 8q .. 8q+7      B (32 x 16): col r, k = 8q .. 8q+7
//   D (16 x 16): col r, rows 4q .. 4q+3 (registers 0..3)
//
// Layers are computed transposed, H^T = W^T X^T: A is the weights, B a band of
// 16 samples.  D then holds 4 features of a sample per lane and tile, and two
// lane swaps per register pair make it the next layer's B (next_operand), so
// activations pass from layer to layer in registers.  Products and their order
// in k are those of X W.
//
// Kernels: forward (weights in registers); training (k_mlp_backprop: forward, loss
// gradient and back, k_mlp_wgrad: weight gradients by chunks of 1024 rows); reduce + Adam.  Loss: relative L2,
// sum_c (p_c - t_c)^2 / (sg(p_c)^2 + 0.01) / N (Mueller et al. 2021).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "objects.h"
#include "wave.h"

namespace solhip {

namespace {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kOut = 3;
constexpr int kHidden = 4;           // layers 0..3 are 64x64 + ReLU, layer 4 is 64x16 linear
constexpr uint32_t kP = 4 * 4096 + 64 * 16;
constexpr int kMlpBlock = 256;       // 4 waves

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf16x8 zero8()
{
    bf16x8 z;
    for (int j = 0; j < 8; ++j) z[j] = (bf16)0.0f;
    return z;
}

constexpr uint32_t kWeights = 4 * 4096 + 16 * 64;   // of either BF16 layout

__device__ __forceinline__ uint32_t wt_offset(int l, int n) { return (uint32_t)l * 4096u + (uint32_t)n * 64u; }

// tiles 2h and 2h + 1 of a layer's output (BF16 x 4 each: features 16 nt + 4q ..
// 4q+3 of sample r) as half h of the next layer's B operand (features 32h + 8q
// .. 8q+7).  With the tiles' rows of 16 lanes a0 a1 a2 a3 and b0 b1 b2 b3, the
// operand's first half is a0 a2 b0 b2 and its second a1 a3 b1 b3: swap a's upper 32
// lanes with b's lower, then a's odd rows with b's even ones.
__device__ __forceinline__ bf16x8 next_operand(bf16x4 ta, bf16x4 tb)
{
    const u32x2 a = __builtin_bit_cast(u32x2, ta), b = __builtin_bit_cast(u32x2, tb);
    u32x4 o;
    for (int k = 0; k < 2; ++k) {
        const auto s = __builtin_amdgcn_permlane32_swap(a[k], b[k], false, false);
        const auto t = __builtin_amdgcn_permlane16_swap(s[0], s[1], false, false);
        o[k] = t[0];
        o[2 + k] = t[1];
    }
    return __builtin_bit_cast(bf16x8, o);
}

// ReLU and rounding of an accumulator tile
__device__ __forceinline__ bf16x4 relu4(f32x4 acc)
{
    bf16x4 v;
    for (int i = 0; i < 4; ++i) v[i] = (bf16)fmaxf(acc[i], 0.0f);
    return v;
}

struct FwdArgs {
    const bf16 *x;          // N x 64
    uint32_t n;
    const uint32_t *n_dev;  // if set, N is read from device memory (at most n)
    const bf16 *wt;         // forward layout
    float4 *y;              // N outputs (x, y, z written), or null
    // cache-query epilogue: st1[rec.path].xyz += rec.T * max(y, 0)
    const CacheQuery *qrec;
    float4 *st1;
};

// Forward: each wave keeps all weights in registers (34 operands, 136 VGPRs) and
// streams bands of 16 rows, kFwdBands at a time, the next ones' loads issued
// before the current ones' layers.  Bound by the 140 B per row it moves.
// 1M rows 139 -> 60 us, 30,000 20 -> 5.7 (weights read from LDS for every tile and
// activations through it before).
constexpr int kFwdBands = 2;

__global__ void __launch_bounds__(kMlpBlock) k_mlp_fwd(FwdArgs A)
{
    __shared__ bf16 wl[kWeights];
    for (uint32_t i = threadIdx.x; i < kWeights / 8; i += kMlpBlock)
        reinterpret_cast<bf16x8 *>(wl)[i] = reinterpret_cast<const bf16x8 *>(A.wt)[i];
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63u, r = lane & 15u, q = lane >> 4, wv = threadIdx.x >> 6;
    bf16x8 w[kHidden][4][2], wo[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int l = 0; l < kHidden; ++l)
#pragma unroll
            for (int nt = 0; nt < 4; ++nt)
                w[l][nt][h] = *reinterpret_cast<const bf16x8 *>(wl + wt_offset(l, nt * 16 + (int)r) + 32 * h + 8 * q);
        wo[h] = *reinterpret_cast<const bf16x8 *>(wl + 4 * 4096 + r * 64 + 32 * h + 8 * q);
    }
    const uint32_t n = A.n_dev ? min(*A.n_dev, A.n) : A.n;
    const uint32_t bands = (n + 15) / 16, stride = gridDim.x * (kMlpBlock / 64) * kFwdBands;
    auto load = [&](uint32_t band, bf16x8 x[2]) {
        const uint32_t row = band * 16 + r;
        const bool in = row < n;
        const bf16 *p = A.x + (uint64_t)(in ? row : 0u) * 64 + 8 * q;
        x[0] = in ? *reinterpret_cast<const bf16x8 *>(p) : zero8();
        x[1] = in ? *reinterpret_cast<const bf16x8 *>(p + 32) : zero8();
    };
    uint32_t band = (blockIdx.x * (kMlpBlock / 64) + wv) * kFwdBands;
    bf16x8 x[kFwdBands][2];
    for (int k = 0; k < kFwdBands; ++k) load(min(band + k, bands), x[k]);
    for (; band < bands; band += stride) {
        bf16x8 nx[kFwdBands][2];
        for (int k = 0; k < kFwdBands; ++k) load(min(band + stride + k, bands), nx[k]);
#pragma unroll
        for (int l = 0; l < kHidden; ++l) {
#pragma unroll
            for (int k = 0; k < kFwdBands; ++k) {
                bf16x4 t[4];
#pragma unroll
                for (int nt = 0; nt < 4; ++nt) {
                    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
                    acc = mfma(w[l][nt][0], x[k][0], acc);
                    acc = mfma(w[l][nt][1], x[k][1], acc);
                    t[nt] = relu4(acc);
                }
                x[k][0] = next_operand(t[0], t[1]);
                x[k][1] = next_operand(t[2], t[3]);
            }
        }
#pragma unroll
        for (int k = 0; k < kFwdBands; ++k) {
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
            acc = mfma(wo[0], x[k][0], acc);
            acc = mfma(wo[1], x[k][1], acc);
            // lanes q == 0 hold the outputs of sample r
            const uint32_t row = (band + k) * 16 + r;
            if (q == 0 && band + k < bands && row < n) {
                if (A.y) {
                    float *o = reinterpret_cast<float *>(A.y + row);
                    o[0] = acc[0];
                    o[1] = acc[1];
                    o[2] = acc[2];
                }
                if (A.qrec) {
                    const CacheQuery rec = A.qrec[row];
                    float *L = reinterpret_cast<float *>(A.st1 + rec.path);
                    for (int c = 0; c < kOut; ++c) L[c] = L[c] + rec.T[c] * fmaxf(acc[c], 0.0f);
                }
            }
            x[k][0] = nx[k][0];
            x[k][1] = nx[k][1];
        }
    }
}

struct TrainArgs {
    const bf16 *x;              // the slab's rows, 64 wide
    const float4 *target;       // their targets (x, y, z, -)
    uint32_t n;                 // rows of the slab
    float invn;                 // 1 / rows of the whole batch
    const bf16 *wt, *wb;        // forward / backward layout
    bf16 *frags;                // operands of the weight gradients (below)
    float *loss;                // [gridDim.x]: the workgroups' loss
};

// Training in two kernels: k_mlp_backprop runs every row forward and back and
// stores the operands of the weight gradients X^T dZ; k_mlp_wgrad sums them
// over chunks of kChunk rows, in row order in one accumulator, and k_mlp_adam adds the
// chunks one after the other.  FP32 sums depend on their order and training
// carries the difference into every later weight, so the order is fixed by the rows
// alone, not by how many workgroups there are.
//
// Operands, per block of 32 rows: 5 x 4 tiles of layer inputs, then 4 x 4 + 1 tiles of
// output gradients, each 16 features x 32 rows as one wave's MFMA operand (lane
// (r, q): feature r, rows 8q .. 8q+7, 16 B): k_mlp_wgrad reads 1 KB a
// load, nothing twice but by the waves that share an operand.
constexpr uint32_t kChunk = 1024;              // rows per partial sum
constexpr uint32_t kFrag = 512;                // elements of an operand
constexpr uint32_t kFragsX = 5 * 4, kFrags = kFragsX + 4 * 4 + 1;   // per 32 rows
// rows whose operands are in memory at a time: 151 MB, within the last-level cache
// (300,001 rows 160 us a step; 180 and 303 with slabs of 64 and 32 chunks, whose launches do not
// fill the GPU)
constexpr uint32_t kSlab = 128 * kChunk;
constexpr uint32_t kRow = 64 + 8;              // row stride of the weights in LDS, in elements
constexpr int kBackBlock = 1024, kBackWaves = kBackBlock / 64;

struct TrainLds {
    bf16 wt[(4 * 64 + 16) * kRow];             // forward layout: row = output, 64 inputs
    bf16 wb[4 * 64 * kRow];                    // backward layout: row = input, 64 outputs
    bf16 wb4[64 * 24];                         // output layer: row = input, 16 outputs (padded to 24)
    bf16 turn[kBackWaves][64 * 24];            // a wave's values of its 16 rows: row = feature
    float loss[kBackWaves];
};

// A wave per band of 16 rows, 16 waves per workgroup (4 per SIMD: a band is a chain of
// nine dependent layers), weights in LDS in both layouts, rows padded to 36
// dwords.  A layer's values pass to the next in registers and, turned to
// feature-major through the wave's own LDS, to memory: no barrier after the
// weights are loaded.  65,536 rows 19 us, of 78 MB written.  A step of training (microseconds
// at 1024, 65,536, 300,001 rows): 26, 41, 160; with activations and gradients written row by
// row in three kernels, in the same order of sums, 60, 161, 490.  One kernel that kept
// the weight gradients in registers took 18, 43, 125, but summed tiles of 64 rows by
// workgroup: the weights after 5 steps differed by 2e-4 of their outputs.
__global__ void __launch_bounds__(kBackBlock) k_mlp_backprop(TrainArgs A)
{
    extern __shared__ uint4 lds_raw[];
    TrainLds &S = *reinterpret_cast<TrainLds *>(lds_raw);
    const uint32_t tid = threadIdx.x, lane = tid & 63u, r = lane & 15u, q = lane >> 4, wv = tid >> 6;
    // weights: rows of 64 (8 x 16 B), padded
    for (uint32_t i = tid; i < (4 * 64 + 16) * 8; i += kBackBlock)
        *reinterpret_cast<bf16x8 *>(S.wt + (i >> 3) * kRow + (i & 7u) * 8) = reinterpret_cast<const bf16x8 *>(A.wt)[i];
    for (uint32_t i = tid; i < 4 * 64 * 8; i += kBackBlock)
        *reinterpret_cast<bf16x8 *>(S.wb + (i >> 3) * kRow + (i & 7u) * 8) = reinterpret_cast<const bf16x8 *>(A.wb)[i];
    for (uint32_t i = tid; i < 64 * 2; i += kBackBlock)
        *reinterpret_cast<bf16x8 *>(S.wb4 + (i >> 1) * 24 + (i & 1u) * 8) =
            reinterpret_cast<const bf16x8 *>(A.wb + 4 * 4096)[i];
    float lsum = 0.0f;
    bf16 *T = S.turn[wv];
    // D-layout values (features 16 nt + 4q + i of row r of the band) into feature-major rows
    auto put = [&](int nt, bf16x4 v) {
#pragma unroll
        for (int i = 0; i < 4; ++i) T[(nt * 16 + 4 * q + i) * 24 + r] = v[i];
    };
    // features 32 p + lane % 32: 8 rows a lane, 2 x 512 B a wave, as the band's half of two operands
    const uint32_t feat = ((lane >> 5) << 4) + r, half = (lane >> 4) & 1u;
    __syncthreads();
    const uint32_t bands = (A.n + 31) / 32 * 2;   // whole blocks of 32 rows: rows from n on are zeros
    for (uint32_t band = blockIdx.x * kBackWaves + wv; band < bands; band += gridDim.x * kBackWaves) {
        bf16 *out = A.frags + (uint64_t)(band >> 1) * (kFrags * kFrag) + (2 * (band & 1u) + half) * 128 + r * 8;
        // the turned values of `tiles` feature tiles as operands at `at`
        auto store = [&](uint32_t at, int tiles) {
            wave_lds_sync();
            for (int p = 0; p < tiles; p += 2)
                if (p + (int)(lane >> 5) < tiles)
                    *reinterpret_cast<bf16x8 *>(out + (at + p + (lane >> 5)) * kFrag) =
                        *reinterpret_cast<const bf16x8 *>(T + (16 * p + feat) * 24 + 8 * half);
            wave_lds_sync();
        };
        const uint32_t row = band * 16 + r;
        const bool in = row < A.n;
        const bf16 *xp = A.x + (uint64_t)(in ? row : 0u) * 64 + 8 * q;
        bf16x8 x0 = in ? *reinterpret_cast<const bf16x8 *>(xp) : zero8();
        bf16x8 x1 = in ? *reinterpret_cast<const bf16x8 *>(xp + 32) : zero8();
        const float4 tg = in && q == 0 ? A.target[row] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            T[(8 * q + j) * 24 + r] = x0[j];
            T[(32 + 8 * q + j) * 24 + r] = x1[j];
        }
        store(0, 4);
        // forward; bit 4 nt + i of mask[l]: the lane's value of layer l's output is positive
        uint32_t mask[kHidden];
#pragma unroll
        for (int l = 0; l < kHidden; ++l) {
            bf16x4 t[4];
            uint32_t mk = 0;
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) {
                const bf16 *w = S.wt + (l * 64 + nt * 16 + (int)r) * kRow + 8 * q;
                f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
                acc = mfma(*reinterpret_cast<const bf16x8 *>(w), x0, acc);
                acc = mfma(*reinterpret_cast<const bf16x8 *>(w + 32), x1, acc);
                t[nt] = relu4(acc);
#pragma unroll
                for (int i = 0; i < 4; ++i) mk |= (float)t[nt][i] > 0.0f ? 1u << (4 * nt + i) : 0u;
                put(nt, t[nt]);
            }
            mask[l] = mk;
            store(4 * (l + 1), 4);
            x0 = next_operand(t[0], t[1]);
            x1 = next_operand(t[2], t[3]);
        }
        f32x4 y = {0.0f, 0.0f, 0.0f, 0.0f};
        {
            const bf16 *w = S.wt + (4 * 64 + r) * kRow + 8 * q;
            y = mfma(*reinterpret_cast<const bf16x8 *>(w), x0, y);
            y = mfma(*reinterpret_cast<const bf16x8 *>(w + 32), x1, y);
        }
        // output gradient: lanes q == 0, k = 0..2 of the next operand
        bf16x8 g0 = zero8(), g1 = zero8();
        if (q == 0 && in) {
            const float tc[3] = {tg.x, tg.y, tg.z};
#pragma unroll
            for (int c = 0; c < kOut; ++c) {
                const float den = y[c] * y[c] + 0.01f, d = y[c] - tc[c];
                lsum += d * d / den * A.invn;
                g0[c] = (bf16)(2.0f * d / den * A.invn);
            }
        }
        put(0, bf16x4{g0[0], g0[1], g0[2], g0[3]});   // zeros but for outputs 0..2
        store(kFragsX + 16, 1);
        // back through layer 4 (k = 16 outputs, padded to 32), then 3..1
#pragma unroll
        for (int l = kHidden; l >= 1; --l) {
            bf16x4 t[4];
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) {
                f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
                if (l == kHidden) {
                    const bf16x8 w = q < 2 ? *reinterpret_cast<const bf16x8 *>(S.wb4 + (nt * 16 + r) * 24 + 8 * q) : zero8();
                    acc = mfma(w, g0, acc);
                } else {
                    const bf16 *w = S.wb + (l * 64 + nt * 16 + (int)r) * kRow + 8 * q;
                    acc = mfma(*reinterpret_cast<const bf16x8 *>(w), g0, acc);
                    acc = mfma(*reinterpret_cast<const bf16x8 *>(w + 32), g1, acc);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) t[nt][i] = (mask[l - 1] >> (4 * nt + i)) & 1u ? (bf16)acc[i] : (bf16)0.0f;
                put(nt, t[nt]);
            }
            store(kFragsX + 4 * (l - 1), 4);
            g0 = next_operand(t[0], t[1]);
            g1 = next_operand(t[2], t[3]);
        }
    }
    for (int off = 32; off > 0; off >>= 1) lsum += __shfl_xor(lsum, off);
    if (lane == 0) S.loss[wv] = lsum;
    __syncthreads();
    if (tid == 0) {
        float l = 0.0f;
        for (int w = 0; w < kBackWaves; ++w) l += S.loss[w];
        A.loss[blockIdx.x] = l;
    }
}

// Weight gradients of one chunk and layer: X^T (rows = inputs) times dZ (rows =
// outputs), k = the chunk's rows in order.  Wave w: input features 16w .. 16w+15.
// Bound by the latency of its 32 dependent blocks of 32 rows, 8 of them in flight
// (65,536 rows 13.4 us, 15.2 with the loads where the compiler puts them).
constexpr int kStages = 8;

template <int TILES>
__device__ __forceinline__ void wgrad(const bf16 *x, const bf16 *d, uint32_t steps, f32x4 acc[TILES])
{
    constexpr uint32_t stride = kFrags * kFrag;
    uint32_t s = 0;
    for (; s + kStages <= steps; s += kStages) {
        bf16x8 a[kStages], b[kStages][TILES];
#pragma unroll
        for (int j = 0; j < kStages; ++j) {
            a[j] = *reinterpret_cast<const bf16x8 *>(x + (uint64_t)(s + j) * stride);
#pragma unroll
            for (int t = 0; t < TILES; ++t)
                b[j][t] = *reinterpret_cast<const bf16x8 *>(d + (uint64_t)(s + j) * stride + t * kFrag);
        }
        __builtin_amdgcn_sched_barrier(0);   // all loads first: the compiler would spread them to save registers
#pragma unroll
        for (int j = 0; j < kStages; ++j)
#pragma unroll
            for (int t = 0; t < TILES; ++t) acc[t] = mfma(a[j], b[j][t], acc[t]);
    }
    for (; s < steps; ++s) {
        const bf16x8 a = *reinterpret_cast<const bf16x8 *>(x + (uint64_t)s * stride);
#pragma unroll
        for (int t = 0; t < TILES; ++t)
            acc[t] = mfma(a, *reinterpret_cast<const bf16x8 *>(d + (uint64_t)s * stride + t * kFrag), acc[t]);
    }
}

// grid (chunks of the slab, 5 layers); partials: [chunks of the slab][kP]
__global__ void __launch_bounds__(kMlpBlock) k_mlp_wgrad(const bf16 *frags, uint32_t blocks32, float *partials)
{
    const uint32_t lane = threadIdx.x & 63u, r = lane & 15u, q = lane >> 4, wv = threadIdx.x >> 6;
    const uint32_t layer = blockIdx.y, first = blockIdx.x * (kChunk / 32), steps = min(kChunk / 32, blocks32 - first);
    const bf16 *base = frags + (uint64_t)first * (kFrags * kFrag) + lane * 8;
    const bf16 *x = base + (4 * layer + wv) * kFrag, *d = base + (kFragsX + 4 * layer) * kFrag;
    float *P = partials + (uint64_t)blockIdx.x * kP + layer * 4096;
    f32x4 acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if (layer < (uint32_t)kHidden) {
        wgrad<4>(x, d, steps, acc);
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) P[(wv * 16 + 4 * q + i) * 64 + t * 16 + r] = acc[t][i];
    } else {
        wgrad<1>(x, d, steps, acc);
#pragma unroll
        for (int i = 0; i < 4; ++i) P[(wv * 16 + 4 * q + i) * 16 + r] = acc[0][i];
    }
}

struct AdamArgs {
    const float *partials;
    uint32_t nchunks;
    const float *loss_parts;
    uint32_t nloss;
    float *loss;
    float *w, *m, *v;
    bf16 *wt, *wb;
    float *grad_out;   // optional: the summed gradient
    float lr, b1, b2, eps, c1, c2;   // c1 = 1 - b1^t, c2 = 1 - b2^t
    uint32_t update;
};

__device__ __forceinline__ bool padded(uint32_t p) { return p >= 16384 && ((p - 16384) & 15u) >= (uint32_t)kOut; }

__device__ __forceinline__ void write_bf16(bf16 *wt, bf16 *wb, uint32_t p, float w)
{
    const bf16 h = (bf16)w;
    wb[p] = h;
    if (p < 16384) {
        const uint32_t l = p >> 12, k = (p >> 6) & 63u, n = p & 63u;
        wt[l * 4096 + n * 64 + k] = h;
    } else {
        const uint32_t k = (p - 16384) >> 4, n = (p - 16384) & 15u;
        wt[16384 + n * 64 + k] = h;
    }
}

// Adds the chunks' partial gradients one after the other (64 parameters per
// block; 4 threads each fetch kAdamChunks chunks at a time into LDS, one adds) and
// applies Adam; block 0 also sums the loss.
constexpr uint32_t kAdamChunks = 64;

__global__ void __launch_bounds__(256) k_mlp_adam(AdamArgs A)
{
    __shared__ float s_part[kAdamChunks][64], s_loss[256];
    const uint32_t j = threadIdx.x & 63u, g = threadIdx.x >> 6, p = blockIdx.x * 64 + j;
    float gr = 0.0f;
    for (uint32_t c0 = 0; c0 < A.nchunks; c0 += kAdamChunks) {
        const uint32_t m = min(kAdamChunks, A.nchunks - c0);
#pragma unroll
        for (uint32_t k = 0; k < kAdamChunks / 4; ++k) {
            const uint32_t c = 4 * k + g;
            if (c < m) s_part[c][j] = A.partials[(uint64_t)(c0 + c) * kP + p];
        }
        __syncthreads();
        if (g == 0) {
#pragma unroll 8
            for (uint32_t c = 0; c < m; ++c) gr += s_part[c][j];
        }
        __syncthreads();
    }
    if (blockIdx.x == 0) {   // block-uniform
        float l = 0.0f;
        for (uint32_t c = threadIdx.x; c < A.nloss; c += 256) l += A.loss_parts[c];
        s_loss[threadIdx.x] = l;
        __syncthreads();
        for (uint32_t h = 128; h > 0; h >>= 1) {
            if (threadIdx.x < h) s_loss[threadIdx.x] += s_loss[threadIdx.x + h];
            __syncthreads();
        }
        if (threadIdx.x == 0) *A.loss = s_loss[0];
    }
    if (g != 0) return;
    if (padded(p)) gr = 0.0f;
    if (A.grad_out) A.grad_out[p] = gr;
    if (!A.update) return;
    const float m = A.b1 * A.m[p] + (1.0f - A.b1) * gr;
    const float v = A.b2 * A.v[p] + (1.0f - A.b2) * gr * gr;
    A.m[p] = m;
    A.v[p] = v;
    float w = A.w[p];
    if (!padded(p)) w -= A.lr * (m / A.c1) / (sqrtf(v / A.c2) + A.eps);
    A.w[p] = w;
    write_bf16(A.wt, A.wb, p, w);
}
static_assert(kP % 64 == 0, "k_mlp_adam: 64 parameters per block");

__global__ void k_mlp_sync_bf16(const float *w, bf16 *wt, bf16 *wb)
{
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < kP) write_bf16(wt, wb, p, w[p]);
}

int mlp_status(const char *what)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error(std::string(what) + " launch: " + hipGetErrorString(e));
        return SOLHIP_ERROR_DEVICE;
    }
    return 0;
}

}  // namespace

struct Mlp : Obj {
    DevBuf w, m, v, wt, wb, frags, partials, loss, loss_parts, grad;
    float lr = 1e-2f, b1 = 0.9f, b2 = 0.99f, eps = 1e-8f;
    uint32_t step = 0, ncu = 256;
    void release_all()
    {
        for (DevBuf *b : {&w, &m, &v, &wt, &wb, &frags, &partials, &loss, &loss_parts, &grad}) b->release();
    }
    // blocks of 4 waves that cover the bands of n rows, two per CU at most
    uint32_t forward_blocks(uint32_t n) const
    {
        const uint32_t per_block = 16u * kFwdBands * (kMlpBlock / 64);
        return std::max(1u, std::min((n + per_block - 1) / per_block, ncu * 2));
    }
    int forward(hipStream_t s, const bf16 *x, uint32_t n, float4 *y)
    {
        FwdArgs a;
        std::memset(&a, 0, sizeof(a));
        a.x = x;
        a.n = n;
        a.wt = (const bf16 *)wt.ptr;
        a.y = y;
        hipLaunchKernelGGL(k_mlp_fwd, dim3(forward_blocks(n)), dim3(kMlpBlock), 0, s, a);
        return mlp_status("mlp forward");
    }
    // loss and its gradient on (x, target), applied by Adam when update
    int fit(hipStream_t s, const bf16 *x, const float4 *target, uint32_t n, bool update, float *grad_host)
    {
        const uint32_t chunks = (n + kChunk - 1) / kChunk, slabs = (n + kSlab - 1) / kSlab;
        const uint64_t block_bytes = kFrags * kFrag * sizeof(bf16), rows = std::min(n, kSlab);
        if (partials.reserve((uint64_t)chunks * kP * 4) || frags.reserve((rows + 31) / 32 * block_bytes) ||
            loss_parts.reserve((uint64_t)slabs * ncu * 4))
            return SOLHIP_ERROR_OUT_OF_MEMORY;
        uint32_t nloss = 0;
        for (uint32_t k = 0; k < slabs; ++k) {
            const uint64_t row0 = (uint64_t)k * kSlab;
            TrainArgs b;
            b.x = x + row0 * 64;
            b.target = target + row0;
            b.n = (uint32_t)std::min<uint64_t>(kSlab, n - row0);
            b.invn = 1.0f / (float)n;
            b.wt = (const bf16 *)wt.ptr;
            b.wb = (const bf16 *)wb.ptr;
            b.frags = (bf16 *)frags.ptr;
            b.loss = (float *)loss_parts.ptr + nloss;
            const uint32_t blocks32 = (b.n + 31) / 32;
            const uint32_t grid = std::min((2 * blocks32 + kBackWaves - 1) / kBackWaves, ncu);
            hipLaunchKernelGGL(k_mlp_backprop, dim3(grid), dim3(kBackBlock), sizeof(TrainLds), s, b);
            hipLaunchKernelGGL(k_mlp_wgrad, dim3((b.n + kChunk - 1) / kChunk, kHidden + 1), dim3(kMlpBlock), 0, s,
                               (const bf16 *)frags.ptr, blocks32,
                               (float *)partials.ptr + (uint64_t)k * (kSlab / kChunk) * kP);
            nloss += grid;
        }
        AdamArgs d;
        d.partials = (const float *)partials.ptr;
        d.nchunks = chunks;
        d.loss_parts = (const float *)loss_parts.ptr;
        d.nloss = nloss;
        d.loss = (float *)loss.ptr;
        d.w = (float *)w.ptr;
        d.m = (float *)m.ptr;
        d.v = (float *)v.ptr;
        d.wt = (bf16 *)wt.ptr;
        d.wb = (bf16 *)wb.ptr;
        d.grad_out = grad_host ? (float *)grad.ptr : nullptr;
        d.update = update ? 1u : 0u;
        if (update) ++step;
        d.lr = lr;
        d.b1 = b1;
        d.b2 = b2;
        d.eps = eps;
        d.c1 = 1.0f - std::pow(b1, (float)std::max(1u, step));
        d.c2 = 1.0f - std::pow(b2, (float)std::max(1u, step));
        hipLaunchKernelGGL(k_mlp_adam, dim3(kP / 64), dim3(256), 0, s, d);
        int rc = mlp_status("mlp training");
        if (rc) return rc;
        if (grad_host) {
            SOLHIP_HIP_CHECK(hipMemcpyAsync(grad_host, grad.ptr, kP * 4, hipMemcpyDeviceToHost, s));
            SOLHIP_HIP_CHECK(hipStreamSynchronize(s));
        }
        return 0;
    }
};

Mlp *mlp_new(Context *c, uint32_t seed, float lr);

int mlp_query(hipStream_t s, Mlp *m, const uint16_t *feat, const uint32_t *n_dev, uint32_t n_max,
              const CacheQuery *qrec, float4 *st1)
{
    FwdArgs a;
    std::memset(&a, 0, sizeof(a));
    a.x = (const bf16 *)feat;
    a.n = n_max;
    a.n_dev = n_dev;
    a.wt = (const bf16 *)m->wt.ptr;
    a.qrec = qrec;
    a.st1 = st1;
    hipLaunchKernelGGL(k_mlp_fwd, dim3(m->forward_blocks(n_max)), dim3(kMlpBlock), 0, s, a);
    return mlp_status("cache query");
}

int mlp_train_dev(hipStream_t s, Mlp *m, const uint16_t *feat, const float4 *target, uint32_t n, uint32_t steps)
{
    if (n == 0) return 0;
    for (uint32_t k = 0; k < steps; ++k) {
        const int rc = m->fit(s, (const bf16 *)feat, target, n, true, nullptr);
        if (rc) return rc;
    }
    return 0;
}

void mlp_delete(Mlp *m)
{
    if (!m) return;
    m->release_all();
    delete m;
}

// He-uniform hidden layers, Glorot-uniform output layer, from a PCG stream
static void init_params(uint32_t seed, std::vector<float> &w)
{
    w.assign(kP, 0.0f);
    uint64_t st = 0x853c49e6748fea9bull ^ ((uint64_t)seed << 1);
    auto next = [&]() {
        st = st * 6364136223846793005ull + 1442695040888963407ull;
        const uint32_t x = (uint32_t)(((st >> 18) ^ st) >> 27), rot = (uint32_t)(st >> 59);
        return ((x >> rot) | (x << ((32 - rot) & 31))) * 0x1p-32f;   // [0, 1)
    };
    const float bh = std::sqrt(6.0f / 64.0f), bo = std::sqrt(6.0f / (64.0f + 3.0f));
    for (uint32_t p = 0; p < 16384; ++p) w[p] = (2.0f * next() - 1.0f) * bh;
    for (uint32_t k = 0; k < 64; ++k)
        for (uint32_t n = 0; n < (uint32_t)kOut; ++n) w[16384 + k * 16 + n] = (2.0f * next() - 1.0f) * bo;
}

static int mlp_sync_from_master(hipStream_t s, Mlp *m)
{
    hipLaunchKernelGGL(k_mlp_sync_bf16, dim3((kP + 255) / 256), dim3(256), 0, s, (const float *)m->w.ptr,
                       (bf16 *)m->wt.ptr, (bf16 *)m->wb.ptr);
    return mlp_status("mlp weights");
}

Mlp *mlp_new(Context *c, uint32_t seed, float lr)
{
    Mlp *m = new Mlp();
    m->kind = Kind::Mlp;
    m->lr = lr;
    m->ncu = c->ncu;
    if (m->w.reserve(kP * 4) || m->m.reserve(kP * 4) || m->v.reserve(kP * 4) || m->wt.reserve(kP * 2) ||
        m->wb.reserve(kP * 2) || m->loss.reserve(256) || m->grad.reserve(kP * 4)) {
        mlp_delete(m);
        set_error("mlp allocation failed");
        return nullptr;
    }
    // 128 KB of the 160 that a workgroup may have
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(k_mlp_backprop), hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)sizeof(TrainLds)) != hipSuccess) {
        mlp_delete(m);
        set_error("the device does not give k_mlp_backprop its LDS");
        return nullptr;
    }
    std::vector<float> w;
    init_params(seed, w);
    std::vector<float> z(kP, 0.0f);
    if (hipMemcpy(m->w.ptr, w.data(), kP * 4, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(m->m.ptr, z.data(), kP * 4, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(m->v.ptr, z.data(), kP * 4, hipMemcpyHostToDevice) != hipSuccess ||
        mlp_sync_from_master(c->stream, m) || hipStreamSynchronize(c->stream) != hipSuccess) {
        mlp_delete(m);
        set_error("mlp initialisation failed");
        return nullptr;
    }
    return m;
}

}  // namespace solhip

using namespace solhip;

namespace {

Mlp *mlp_of(solhip_mlp h) { return get<Mlp>(h, Kind::Mlp); }

}  // namespace

extern "C" {

int32_t solhip_mlp_create(solhip_ctx ctx, uint32_t seed, float learning_rate, solhip_mlp *out)
{
    Context *c = ctx_of(ctx);
    if (!c) return bad_handle("context");
    if (!out || !(learning_rate > 0.0f)) return bad_arg("out / learning_rate");
    Mlp *m = mlp_new(c, seed, learning_rate);
    if (!m) return SOLHIP_ERROR_DEVICE;
    m->ctx = ctx;
    *out = reg(m);
    return SOLHIP_OK;
}

int32_t solhip_mlp_destroy(solhip_ctx ctx, solhip_mlp h)
{
    Context *c = ctx_of(ctx);
    if (!c) return bad_handle("context");
    Mlp *m = static_cast<Mlp *>(unreg(h, Kind::Mlp));
    if (!m) return bad_handle("mlp");
    (void)hipDeviceSynchronize();
    mlp_delete(m);
    return SOLHIP_OK;
}

int32_t solhip_mlp_params(solhip_ctx ctx, solhip_mlp h, float *get_out, const float *set_in)
{
    Context *c = ctx_of(ctx);
    if (!c) return bad_handle("context");
    Mlp *m = mlp_of(h);
    if (!m) return bad_handle("mlp");
    SOLHIP_HIP_CHECK(hipDeviceSynchronize());
    if (set_in) {
        std::vector<float> w(set_in, set_in + kP);
        for (uint32_t p = 16384; p < kP; ++p)
            if (((p - 16384) & 15u) >= (uint32_t)kOut) w[p] = 0.0f;
        SOLHIP_HIP_CHECK(hipMemcpy(m->w.ptr, w.data(), kP * 4, hipMemcpyHostToDevice));
        int rc = mlp_sync_from_master(c->stream, m);
        if (rc) return rc;
        SOLHIP_HIP_CHECK(hipStreamSynchronize(c->stream));
    }
    if (get_out) SOLHIP_HIP_CHECK(hipMemcpy(get_out, m->w.ptr, kP * 4, hipMemcpyDeviceToHost));
    return SOLHIP_OK;
}

static int mlp_io(Context *c, solhip_buffer in, uint64_t in_bytes, solhip_buffer o, uint64_t o_bytes, void **pin,
                  void **po)
{
    Buffer *bi = get<Buffer>(in, Kind::Buffer);
    Buffer *bo = get<Buffer>(o, Kind::Buffer);
    (void)c;
    if (!bi || !bo) return bad_handle("buffer");
    if (bi->bytes < in_bytes || bo->bytes < o_bytes) return bad_arg("buffer too small");
    *pin = bi->ptr;
    *po = bo->ptr;
    return 0;
}

int32_t solhip_mlp_forward(solhip_ctx ctx, solhip_stream st, solhip_mlp h, solhip_buffer in, uint32_t n,
                           solhip_buffer out)
{
    Context *c = ctx_of(ctx);
    if (!c) return bad_handle("context");
    bool ok;
    hipStream_t s = stream_of(c, st, ok);
    if (!ok) return bad_handle("stream");
    Mlp *m = mlp_of(h);
    if (!m) return bad_handle("mlp");
    if (n == 0) return SOLHIP_OK;
    void *pi, *po;
    int rc = mlp_io(c, in, (uint64_t)n * 128, out, (uint64_t)n * 16, &pi, &po);
    if (rc) return rc;
    return m->forward(s, (const bf16 *)pi, n, (float4 *)po);
}

static int32_t mlp_fit(solhip_ctx ctx, solhip_stream st, solhip_mlp h, solhip_buffer in, solhip_buffer target,
                       uint32_t n, uint32_t steps, bool update, float *grad_host, float *loss_out)
{
    Context *c = ctx_of(ctx);
    if (!c) return bad_handle("context");
    bool ok;
    hipStream_t s = stream_of(c, st, ok);
    if (!ok) return bad_handle("stream");
    Mlp *m = mlp_of(h);
    if (!m) return bad_handle("mlp");
    if (n == 0 || steps == 0) return bad_arg("n / steps");
    void *pi, *pt;
    int rc = mlp_io(c, in, (uint64_t)n * 128, target, (uint64_t)n * 16, &pi, &pt);
    if (rc) return rc;
    for (uint32_t k = 0; k < steps; ++k) {
        rc = m->fit(s, (const bf16 *)pi, (const float4 *)pt, n, update, k + 1 == steps ? grad_host : nullptr);
        if (rc) return rc;
    }
    if (loss_out) {
        SOLHIP_HIP_CHECK(hipMemcpyAsync(loss_out, m->loss.ptr, 4, hipMemcpyDeviceToHost, s));
        SOLHIP_HIP_CHECK(hipStreamSynchronize(s));
    }
    return SOLHIP_OK;
}

int32_t solhip_mlp_train(solhip_ctx ctx, solhip_stream st, solhip_mlp h, solhip_buffer in, solhip_buffer target,
                         uint32_t n, uint32_t steps, float *loss)
{
    return mlp_fit(ctx, st, h, in, target, n, steps, true, nullptr, loss);
}

int32_t solhip_mlp_gradient(solhip_ctx ctx, solhip_stream st, solhip_mlp h, solhip_buffer in, solhip_buffer target,
                            uint32_t n, float *grad, float *loss)
{
    if (!grad) return bad_arg("grad");
    return mlp_fit(ctx, st, h, in, target, n, 1, false, grad, loss);
}

}  // extern "C"
