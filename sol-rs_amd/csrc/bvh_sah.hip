// bvh_sah.hip -- binary tree of a fast-trace BLAS build, by binned SAH.
//
// The rules of a split are bvh_logic.h's (sah_scale, sah_bin, sah_choose; the
// host replay builds the same tree from them): 32 centroid bins per axis, the
// split of least A(left) N(left) + A(right) N(right), the first of equals in
// axis and bin order, the range halved in its order without a usable split and
// from depth kSahMedianLevel on; both sides keep their primitives' order.
//
// Node numbering: the internal node that splits leaf positions p | p+1 is
// node p.  Every internal node has its own p, so nothing is allocated, and a
// subtree's nodes are neighbours in memory.  A child's index is known only
// once the child is split, so a task carries its parent link (parent << 1 |
// side) and stores its own index there.
//
// Nodes of more than kSubtree primitives are split level by level over the
// whole GPU: three launches a level (bin, split, partition), each over chunks
// of up to kChunk primitives.  Boxes move with the partition (32 B streams
// from one buffer to the other), so every pass reads contiguous memory; a
// chunk's bins are kept until the split is chosen and then give the chunk's
// left count, so partitioning needs no counting pass.  Every smaller node is finished by
// one workgroup with its boxes in LDS (k_sah_subtree).
//
// One workgroup per node at every level (three passes through an index
// array, a launch and a read-back per level) ran the root of a 2.1M-triangle
// mesh on one CU for 20 ms and spent 55 ms on nodes of a few primitives:
// loading that mesh (build, TLAS, 500 rays, release) 106 -> 5.7 ms; of it the
// tree 3.0 ms, collapse 0.55, the rest allocation and release.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "bvh.h"
#include "bvh_logic.h"
#include "common.h"
#include "wave.h"

namespace solhip {

namespace {

constexpr uint32_t kNoLink = 0xFFFFFFFFu;      // link of the root
constexpr uint32_t kSubtree = 1024;            // largest node finished in LDS
constexpr uint32_t kChunk = 4096;              // primitives per workgroup of a large node ...
constexpr uint32_t kMaxChunks = 512;           // ... unless it would have more chunks than this
constexpr int kBinBlock = 256, kSplitBlock = 512, kSubBlock = 256;
constexpr uint32_t kBins = 3 * kSahBins;       // bins of all axes
constexpr uint32_t kBinWords = 7 * kBins;      // word k * kBins + 32 a + b: k = 0 count, 1-3 box min, 4-6 box max
constexpr uint32_t kPartWords = kBinWords + 8; // a chunk's bins, then its box (3 min, 3 max, 2 unused)
constexpr uint32_t kMaxSahLevels = 96;         // kSahMedianLevel + 31 halvings, and spare
// count words: tasks and chunks of each level, small tasks
constexpr uint32_t kCountSmall = 2 * (kMaxSahLevels + 1), kCountWords = kCountSmall + 2;
static_assert(kCountWords <= kPinnedWords, "counts are read back through DevScratch::pinned");
static_assert(kSahBins == 32, "half-wave scans");

struct SplitRec {
    int axis, bin;
    uint32_t nleft;
    uint32_t child[2];   // next-level task of each side (kNoLink: none)
};

struct Work {
    float4 *prim[2];        // box min (w: primitive), box max; by position; ping-pong by level
    uint4 *tasks[2];        // first position, count, link, first chunk
    uint32_t *cbounds[2];   // per task: centroid min, max (ordered integers)
    uint2 *chunks[2];       // task, index within the task
    uint4 *small;           // first position, count, link, level << 1 | buffer
    uint32_t *parts;        // per chunk: kPartWords
    uint32_t *lbase;        // per chunk: the node's left primitives before it
    SplitRec *splits;       // per task
    uint32_t *counts;
    uint32_t *left, *right, *rfirst, *ncount, *vals, *wsrc, *err;
    float4 *nbox;
    uint32_t n, cap_tasks, cap_chunks, cap_small;
};

__host__ __device__ inline uint32_t cap_tasks(uint32_t n) { return n / kSubtree + 1; }
__host__ __device__ inline uint32_t cap_chunks(uint32_t n) { return n / kChunk + 2 * cap_tasks(n) + 1; }

__device__ __forceinline__ uint32_t chunk_count(uint32_t cnt)
{
    return min((cnt + kChunk - 1) / kChunk, kMaxChunks);
}
__device__ __forceinline__ uint32_t chunk_size(uint32_t cnt, uint32_t chunks) { return (cnt + chunks - 1) / chunks; }

__device__ __forceinline__ void centroid(float4 l, float4 h, float c[3])
{
    c[0] = 0.5f * l.x + 0.5f * h.x;
    c[1] = 0.5f * l.y + 0.5f * h.y;
    c[2] = 0.5f * l.z + 0.5f * h.z;
}

// bin frame from centroid bounds (ordered integers)
__device__ __forceinline__ void bin_frame(const uint32_t *cb, float cmin[3], float scale[3])
{
    for (int a = 0; a < 3; ++a) {
        cmin[a] = ord2f(cb[a]);
        scale[a] = sah_scale(ord2f(cb[3 + a]) - cmin[a]);
    }
}

__device__ __forceinline__ void clear_bins(uint32_t *bins, uint32_t t, uint32_t threads)
{
    for (uint32_t w = t; w < kBinWords; w += threads)
        bins[w] = w < kBins ? 0u : (w < 4 * kBins ? f2ord(INFINITY) : f2ord(-INFINITY));
}

// One primitive per lane into the bins (LDS); every lane of the wave calls
// it.  Neighbours mostly share a bin: a wave whose lanes all fall in one bin
// reduces in registers and updates it once.
__device__ __forceinline__ void bin_wave(uint32_t *bins, bool valid, float4 l, float4 h, const float cmin[3],
                                         const float scale[3])
{
    float c[3];
    centroid(l, h, c);
    const uint32_t box[6] = {valid ? f2ord(l.x) : 0xFFFFFFFFu, valid ? f2ord(l.y) : 0xFFFFFFFFu,
                             valid ? f2ord(l.z) : 0xFFFFFFFFu, valid ? f2ord(h.x) : 0u,
                             valid ? f2ord(h.y) : 0u,           valid ? f2ord(h.z) : 0u};
    const uint64_t vmask = __ballot(valid);
    if (vmask == 0) return;
    const int first = __ffsll((unsigned long long)vmask) - 1;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (!(scale[a] > 0.0f)) continue;   // uniform
        const int b = sah_bin(c[a], cmin[a], scale[a]);
        const int b0 = __builtin_amdgcn_readlane(b, first);
        if (__ballot(valid && b != b0) == 0) {
            uint32_t r[6];
            for (int k = 0; k < 6; ++k) r[k] = k < 3 ? wave_min(box[k]) : wave_max(box[k]);
            if ((threadIdx.x & 63u) == 0) {
                uint32_t *at = bins + a * kSahBins + b0;
                atomicAdd(at, (uint32_t)__popcll(vmask));
                for (int k = 0; k < 3; ++k) {
                    atomicMin(at + (1 + k) * kBins, r[k]);
                    atomicMax(at + (4 + k) * kBins, r[3 + k]);
                }
            }
        } else if (valid) {
            uint32_t *at = bins + a * kSahBins + b;
            atomicAdd(at, 1u);
            for (int k = 0; k < 3; ++k) {
                atomicMin(at + (1 + k) * kBins, box[k]);
                atomicMax(at + (4 + k) * kBins, box[3 + k]);
            }
        }
    }
}

__device__ __forceinline__ float ord_area(const uint32_t lo[3], const uint32_t hi[3])
{
    const float l[3] = {ord2f(lo[0]), ord2f(lo[1]), ord2f(lo[2])}, h[3] = {ord2f(hi[0]), ord2f(hi[1]), ord2f(hi[2])};
    return half_area3(l, h);
}

// Best split of axes a0 and a0 + 1 (one per half wave, a lane per bin), the
// first strict minimum in axis and bin order: its ordered cost in the result
// (0xFFFFFFFF: none) and the split in sp.  All lanes call it.
__device__ __forceinline__ uint32_t split_axes(const uint32_t *bins, int a0, const float scale[3], SahSplit &sp)
{
    const uint32_t lane = threadIdx.x & 63u, b = lane & 31u;
    const int a = a0 + (int)(lane >> 5);
    const bool usable = a < 3 && (a == 0 ? scale[0] : (a == 1 ? scale[1] : scale[2])) > 0.0f;
    auto add = [](uint32_t x, uint32_t y) { return x + y; };
    auto mn = [](uint32_t x, uint32_t y) { return min(x, y); };
    auto mx = [](uint32_t x, uint32_t y) { return max(x, y); };
    // bins 0..b, and (lanes in reverse bin order) bins 31-b..31
    uint32_t cnt[2], lo[2][3], hi[2][3];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const uint32_t *at = bins + (usable ? a : 0) * kSahBins + (r ? 31u - b : b);
        cnt[r] = half_scan(at[0], 0u, add);
        for (int k = 0; k < 3; ++k) {
            lo[r][k] = half_scan(at[(1 + k) * kBins], 0xFFFFFFFFu, mn);
            hi[r][k] = half_scan(at[(4 + k) * kBins], 0u, mx);
        }
    }
    const float area_r = cnt[1] ? ord_area(lo[1], hi[1]) : 0.0f;
    const int src = (int)((lane & 32u) + (b < 31u ? 30u - b : 0u));   // the lane that holds bins b+1..31
    const uint32_t rc = __shfl(cnt[1], src);
    const float ra = __shfl(area_r, src);
    uint32_t key = 0xFFFFFFFFu;
    if (usable && b < 31u && cnt[0] && rc) {
        const float cost = ord_area(lo[0], hi[0]) * (float)cnt[0] + ra * (float)rc;
        if (cost < INFINITY) key = f2ord(cost);
    }
    const uint32_t best = wave_min(key);
    if (best != 0xFFFFFFFFu) {
        const int win = __ffsll((unsigned long long)__ballot(key == best)) - 1;
        sp.axis = a0 + (win >> 5);
        sp.bin = win & 31;
        sp.nleft = (uint32_t)__builtin_amdgcn_readlane((int)cnt[0], win);
    }
    return best;
}

// node `id` of range [lo, lo + cnt) hangs below its link
__device__ __forceinline__ void place_node(const Work &W, uint32_t id, uint32_t lo, uint32_t cnt, uint32_t link,
                                           float4 bl, float4 bh)
{
    W.rfirst[id] = lo;
    W.ncount[id] = cnt;
    W.nbox[2ull * id] = bl;
    W.nbox[2ull * id + 1] = bh;
    if (link == kNoLink) W.wsrc[0] = id;
    else ((link & 1u) ? W.right : W.left)[link >> 1] = id;
}

// the leaf at position pos, a child of node `parent`
__device__ __forceinline__ void place_leaf(const Work &W, uint32_t pos, uint32_t prim, float4 bl, float4 bh)
{
    W.vals[pos] = prim;
    W.nbox[2ull * (W.n - 1u + pos)] = bl;
    W.nbox[2ull * (W.n - 1u + pos) + 1] = bh;
    W.ncount[W.n - 1u + pos] = 1u;
}

// ---- nodes of more than kSubtree primitives, level by level ---------------

__global__ void k_sah_root(Work W, const uint32_t *bounds)
{
    const uint32_t t = threadIdx.x;
    const bool big = W.n > kSubtree;
    const uint32_t nch = chunk_count(W.n);
    for (uint32_t k = t; k < kCountWords; k += blockDim.x)
        W.counts[k] = k == 0 ? (big ? 1u : 0u) : k == 1 ? (big ? nch : 0u) : k == kCountSmall ? (big ? 0u : 1u) : 0u;
    if (t == 0) {
        if (big) W.tasks[0][0] = make_uint4(0u, W.n, kNoLink, 0u);
        else W.small[0] = make_uint4(0u, W.n, kNoLink, 0u);
    }
    if (big) {
        if (t < 6) W.cbounds[0][t] = bounds[t];
        for (uint32_t k = t; k < nch; k += blockDim.x) W.chunks[0][k] = make_uint2(0u, k);
    }
}

// bins and box of every chunk of the level.  Bound by the 32 B per primitive
// it reads (top levels) and by the LDS updates of waves that span many bins.
__global__ void __launch_bounds__(kBinBlock) k_sah_bin(Work W, uint32_t level)
{
    __shared__ uint32_t bins[kBinWords];
    __shared__ uint32_t s_box[6];
    const uint32_t cur = level & 1u, tid = threadIdx.x;
    if (blockIdx.x >= min(W.counts[2 * level + 1], W.cap_chunks)) return;
    const uint2 ck = W.chunks[cur][blockIdx.x];
    const uint4 t = W.tasks[cur][ck.x];
    const uint32_t size = chunk_size(t.y, chunk_count(t.y));
    const uint32_t begin = min(t.x + ck.y * size, t.x + t.y), end = min(begin + size, t.x + t.y);
    float cmin[3], scale[3];
    bin_frame(W.cbounds[cur] + 6ull * ck.x, cmin, scale);
    if (level >= kSahMedianLevel) scale[0] = scale[1] = scale[2] = 0.0f;
    clear_bins(bins, tid, kBinBlock);
    if (tid < 6) s_box[tid] = tid < 3 ? 0xFFFFFFFFu : 0u;
    __syncthreads();
    uint32_t box[6] = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0u, 0u, 0u};
    const float4 *prim = W.prim[cur];
    for (uint32_t base = begin; base < end; base += kBinBlock) {
        const uint32_t i = base + tid;
        const bool valid = i < end;
        float4 l = make_float4(0.0f, 0.0f, 0.0f, 0.0f), h = l;
        if (valid) {
            l = prim[2ull * i];
            h = prim[2ull * i + 1];
            box[0] = min(box[0], f2ord(l.x));
            box[1] = min(box[1], f2ord(l.y));
            box[2] = min(box[2], f2ord(l.z));
            box[3] = max(box[3], f2ord(h.x));
            box[4] = max(box[4], f2ord(h.y));
            box[5] = max(box[5], f2ord(h.z));
        }
        bin_wave(bins, valid, l, h, cmin, scale);
    }
    for (int k = 0; k < 6; ++k) {
        const uint32_t r = k < 3 ? wave_min(box[k]) : wave_max(box[k]);
        if ((tid & 63u) == 0) {
            if (k < 3) atomicMin(&s_box[k], r);
            else atomicMax(&s_box[k], r);
        }
    }
    __syncthreads();
    uint32_t *out = W.parts + (uint64_t)blockIdx.x * kPartWords;
    for (uint32_t w = tid; w < kBinWords; w += kBinBlock) out[w] = bins[w];
    if (tid < 8) out[kBinWords + tid] = tid < 6 ? s_box[tid] : 0u;
}

// one workgroup per node of the level: its bins from its chunks', the split,
// the chunks' left offsets, and the children as tasks
__global__ void __launch_bounds__(kSplitBlock) k_sah_split(Work W, uint32_t level)
{
    constexpr uint32_t kQuads = kPartWords / 4, kGroups = kSplitBlock / kQuads;
    __shared__ uint32_t s_bins[kGroups][kPartWords];
    __shared__ SahSplit s_sp[2];
    __shared__ uint32_t s_key[2], s_scan[kSplitBlock / 64], s_child[2][2];
    const uint32_t cur = level & 1u, nxt = cur ^ 1u, tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    if (blockIdx.x >= min(W.counts[2 * level], W.cap_tasks)) return;
    const uint4 t = W.tasks[cur][blockIdx.x];
    const uint32_t lo = t.x, cnt = t.y, nch = chunk_count(cnt), size = chunk_size(cnt, nch);
    auto combine = [](uint32_t w, uint32_t x, uint32_t y) {
        const bool is_min = (w >= kBins && w < 4 * kBins) || (w >= kBinWords && w < kBinWords + 3);
        return w < kBins ? x + y : (is_min ? min(x, y) : max(x, y));
    };
    // thread: 4 words, every kGroups-th chunk
    if (tid < kGroups * kQuads) {
        const uint32_t g = tid / kQuads, q = tid - g * kQuads;
        uint32_t v[4];
        for (int k = 0; k < 4; ++k) {
            const uint32_t w = 4 * q + k;
            const bool is_min = (w >= kBins && w < 4 * kBins) || (w >= kBinWords && w < kBinWords + 3);
            v[k] = is_min ? 0xFFFFFFFFu : 0u;
        }
        const uint4 *part = reinterpret_cast<const uint4 *>(W.parts) + (uint64_t)t.w * kQuads + q;
#pragma unroll 8
        for (uint32_t k = g; k < nch; k += kGroups) {
            const uint4 p = part[(uint64_t)k * kQuads];
            v[0] = combine(4 * q, v[0], p.x);
            v[1] = combine(4 * q + 1, v[1], p.y);
            v[2] = combine(4 * q + 2, v[2], p.z);
            v[3] = combine(4 * q + 3, v[3], p.w);
        }
        for (int k = 0; k < 4; ++k) s_bins[g][4 * q + k] = v[k];
    }
    __syncthreads();
    for (uint32_t w = tid; w < kPartWords; w += kSplitBlock)
        for (uint32_t g = 1; g < kGroups; ++g) s_bins[0][w] = combine(w, s_bins[0][w], s_bins[g][w]);
    __syncthreads();
    float cmin[3], scale[3];
    bin_frame(W.cbounds[cur] + 6ull * blockIdx.x, cmin, scale);
    if (level >= kSahMedianLevel) scale[0] = scale[1] = scale[2] = 0.0f;
    if (wave < 2) {   // wave 0: axes x and y, wave 1: z
        SahSplit sp{-1, 0, cnt / 2};
        const uint32_t key = split_axes(s_bins[0], wave ? 2 : 0, scale, sp);
        if (lane == 0) {
            s_key[wave] = key;
            s_sp[wave] = sp;
        }
    }
    __syncthreads();
    const SahSplit sp = s_key[1] < s_key[0] ? s_sp[1] : s_sp[0];
    const uint32_t nleft = sp.nleft, nright = cnt - nleft, id = lo + nleft - 1u;
    if (nleft == 0u || nleft >= cnt) {   // block-uniform; cannot happen
        if (tid == 0) {
            atomicAdd(W.err, 1u);
            W.splits[blockIdx.x].nleft = 0u;   // k_sah_part leaves the node alone
        }
        return;
    }
    // left primitives of this thread's chunk, and before it
    uint32_t lc = 0;
    if (tid < nch) {
        const uint32_t b0 = min(tid * size, cnt), b1 = min(b0 + size, cnt);
        if (sp.axis >= 0) {
            const uint32_t *c = W.parts + (uint64_t)(t.w + tid) * kPartWords + sp.axis * kSahBins;
            for (int b = 0; b <= sp.bin; ++b) lc += c[b];
        } else {
            lc = min(b1, nleft) - min(b0, nleft);
        }
    }
    uint32_t incl = lc;
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t u = __shfl_up(incl, d);
        if (lane >= (uint32_t)d) incl += u;
    }
    if (lane == 63) s_scan[wave] = incl;
    __syncthreads();
    uint32_t before = 0;
    for (uint32_t w = 0; w < wave; ++w) before += s_scan[w];
    if (tid < nch) W.lbase[t.w + tid] = before + incl - lc;
    if (tid == 0) {
        const uint32_t *bx = s_bins[0] + kBinWords;
        place_node(W, id, lo, cnt, t.z, make_float4(ord2f(bx[0]), ord2f(bx[1]), ord2f(bx[2]), 0.0f),
                   make_float4(ord2f(bx[3]), ord2f(bx[4]), ord2f(bx[5]), 0.0f));
        SplitRec rec{sp.axis, sp.bin, nleft, {kNoLink, kNoLink}};
        for (uint32_t side = 0; side < 2; ++side) {
            const uint32_t start = side ? lo + nleft : lo, m = side ? nright : nleft, link = (id << 1) | side;
            s_child[side][0] = kNoLink;
            if (m == 1u) {
                (side ? W.right : W.left)[id] = W.n - 1u + start;   // the leaf itself: k_sah_part
            } else if (m <= kSubtree) {
                const uint32_t at = atomicAdd(W.counts + kCountSmall, 1u);
                if (at < W.cap_small) W.small[at] = make_uint4(start, m, link, ((level + 1) << 1) | nxt);
                else atomicAdd(W.err, 1u);
            } else {
                const uint32_t at = atomicAdd(W.counts + 2 * (level + 1), 1u), c = chunk_count(m);
                const uint32_t c0 = atomicAdd(W.counts + 2 * (level + 1) + 1, c);
                if (at < W.cap_tasks && c0 + c <= W.cap_chunks) {
                    W.tasks[nxt][at] = make_uint4(start, m, link, c0);
                    rec.child[side] = at;
                    s_child[side][0] = at;
                    s_child[side][1] = c0;
                } else {
                    atomicAdd(W.err, 1u);
                }
            }
        }
        W.splits[blockIdx.x] = rec;
    }
    __syncthreads();
    for (uint32_t side = 0; side < 2; ++side) {
        const uint32_t at = s_child[side][0];
        if (at == kNoLink) continue;
        if (tid < 6) W.cbounds[nxt][6ull * at + tid] = tid < 3 ? 0xFFFFFFFFu : 0u;
        const uint32_t c = chunk_count(side ? nright : nleft);
        for (uint32_t k = tid; k < c; k += kSplitBlock) W.chunks[nxt][s_child[side][1] + k] = make_uint2(at, k);
    }
}

// stable partition of every chunk into the other buffer, and the centroid
// bounds of children that are split at the next level
__global__ void __launch_bounds__(kBinBlock) k_sah_part(Work W, uint32_t level)
{
    constexpr uint32_t kWaves = kBinBlock / 64;
    __shared__ uint32_t s_wave[2][kWaves];
    __shared__ uint32_t s_cb[2][6];
    const uint32_t cur = level & 1u, nxt = cur ^ 1u, tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    if (blockIdx.x >= min(W.counts[2 * level + 1], W.cap_chunks)) return;
    const uint2 ck = W.chunks[cur][blockIdx.x];
    const uint4 t = W.tasks[cur][ck.x];
    const SplitRec sp = W.splits[ck.x];
    const uint32_t lo = t.x, cnt = t.y, size = chunk_size(cnt, chunk_count(cnt));
    const uint32_t begin = min(lo + ck.y * size, lo + cnt), end = min(begin + size, lo + cnt);
    const uint32_t nleft = sp.nleft, nright = cnt - nleft;
    if (nleft == 0u || nleft >= cnt) return;   // block-uniform; counted by k_sah_split
    float cmin[3], scale[3];
    bin_frame(W.cbounds[cur] + 6ull * ck.x, cmin, scale);
    const float cm = sp.axis == 0 ? cmin[0] : (sp.axis == 1 ? cmin[1] : cmin[2]);
    const float sc = sp.axis == 0 ? scale[0] : (sp.axis == 1 ? scale[1] : scale[2]);
    if (tid < 12) s_cb[tid / 6][tid % 6] = tid % 6 < 3 ? 0xFFFFFFFFu : 0u;
    uint32_t cb[2][6];
    for (int s = 0; s < 2; ++s)
        for (int k = 0; k < 6; ++k) cb[s][k] = k < 3 ? 0xFFFFFFFFu : 0u;
    const float4 *in = W.prim[cur];
    float4 *out = W.prim[nxt];
    uint32_t lrun = W.lbase[blockIdx.x], rrun = begin - lo - lrun;
    uint32_t flip = 0;
    for (uint32_t base = begin; base < end; base += kBinBlock, flip ^= 1u) {
        const uint32_t i = base + tid;
        const bool valid = i < end;
        float4 l = make_float4(0.0f, 0.0f, 0.0f, 0.0f), h = l;
        float c[3] = {0.0f, 0.0f, 0.0f};
        bool left = false;
        if (valid) {
            l = in[2ull * i];
            h = in[2ull * i + 1];
            centroid(l, h, c);
            const float ca = sp.axis == 0 ? c[0] : (sp.axis == 1 ? c[1] : c[2]);
            left = sp.axis >= 0 ? sah_bin(ca, cm, sc) <= sp.bin : i - lo < nleft;
        }
        const uint64_t m = __ballot(left);
        if (lane == 0) s_wave[flip][wave] = (uint32_t)__popcll(m);
        __syncthreads();   // (the other half of s_wave is written next, after everyone has passed this one)
        uint32_t woff = 0, total = 0;
        for (uint32_t w = 0; w < kWaves; ++w) {
            woff += w < wave ? s_wave[flip][w] : 0u;
            total += s_wave[flip][w];
        }
        if (valid) {
            const uint32_t lrank = woff + (uint32_t)__popcll(m & ((1ull << lane) - 1ull)), rrank = (i - base) - lrank;
            const uint32_t pos = left ? lo + lrun + lrank : lo + nleft + rrun + rrank;
            if (left ? lrun + lrank < nleft : rrun + rrank < nright) {
                out[2ull * pos] = l;
                out[2ull * pos + 1] = h;
                if ((left ? nleft : nright) == 1u) place_leaf(W, pos, __float_as_uint(l.w), l, h);
            } else {
                atomicAdd(W.err, 1u);
            }
#pragma unroll
            for (int s = 0; s < 2; ++s)
                if (left == (s == 0))
                    for (int k = 0; k < 3; ++k) {
                        cb[s][k] = min(cb[s][k], f2ord(c[k]));
                        cb[s][3 + k] = max(cb[s][3 + k], f2ord(c[k]));
                    }
        }
        lrun += total;
        rrun += min((uint32_t)kBinBlock, end - base) - total;
    }
    __syncthreads();
    for (int s = 0; s < 2; ++s) {
        if (sp.child[s] == kNoLink) continue;   // uniform
        for (int k = 0; k < 6; ++k) {
            const uint32_t r = k < 3 ? wave_min(cb[s][k]) : wave_max(cb[s][k]);
            if (lane == 0) {
                if (k < 3) atomicMin(&s_cb[s][k], r);
                else atomicMax(&s_cb[s][k], r);
            }
        }
    }
    __syncthreads();
    if (tid < 12) {
        const uint32_t s = tid / 6, k = tid % 6, child = sp.child[s];
        if (child != kNoLink) {
            uint32_t *dst = W.cbounds[nxt] + 6ull * child + k;
            if (k < 3) atomicMin(dst, s_cb[s][k]);
            else atomicMax(dst, s_cb[s][k]);
        }
    }
}

// ---- nodes of at most kSubtree primitives: the whole subtree in LDS -------
// One workgroup per subtree.  Nodes of more than kTiny primitives: a wave each,
// level by level, with the wave's own bins.  Smaller ones: 16 lanes each, a
// lane per primitive, to the last leaf: every lane evaluates the split at
// its own primitive's bin (the only bins where the sides change), so
// no bins are needed; the cost of a bin is lower in lanes than in bins up to
// about 16 primitives.
constexpr uint32_t kTiny = 16;
constexpr uint32_t kMaxBigs = kSubtree / (kTiny + 1) + 1;   // disjoint nodes of more than kTiny primitives
constexpr uint32_t kMaxTinies = kSubtree / 2;               // disjoint nodes of at least 2

struct SubtreeLds {
    float box[6][kSubtree];           // by primitive of the subtree
    uint32_t gid[kSubtree];
    uint16_t order[2][kSubtree];      // primitive at each position; ping-pong by level
    uint32_t bins[kSubBlock / 64][kBinWords];
    uint2 big[2][kMaxBigs];           // first position | count << 16, link
    uint2 tiny[kMaxTinies];           // first position | count << 11 | order buffer << 16 | level << 17, link
    uint32_t nbig[2], ntiny;
};
static_assert(sizeof(uint32_t) * 4 * kBinWords >= sizeof(float) * (kSubBlock / 16) * 9 * 16,
              "the tiny phase's exchange area reuses the bins");

__global__ void __launch_bounds__(kSubBlock) k_sah_subtree(Work W)
{
    __shared__ SubtreeLds S;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    constexpr uint32_t kWaves = kSubBlock / 64;
    const uint4 t = W.small[blockIdx.x];
    const uint32_t lo0 = t.x, m = t.y, n = W.n;
    if (m < 2u || m > kSubtree || lo0 > n - m) {   // block-uniform
        if (tid == 0) atomicAdd(W.err, 1u);
        return;
    }
    const uint32_t level0 = t.w >> 1;
    const float4 *prim = W.prim[t.w & 1u] + 2ull * lo0;
    for (uint32_t i = tid; i < m; i += kSubBlock) {
        const float4 l = prim[2 * i], h = prim[2 * i + 1];
        S.box[0][i] = l.x;
        S.box[1][i] = l.y;
        S.box[2][i] = l.z;
        S.box[3][i] = h.x;
        S.box[4][i] = h.y;
        S.box[5][i] = h.z;
        S.gid[i] = __float_as_uint(l.w);
        S.order[0][i] = (uint16_t)i;
    }
    if (tid == 0) {
        S.nbig[0] = m > kTiny ? 1u : 0u;
        S.nbig[1] = 0;
        S.ntiny = m > kTiny ? 0u : 1u;
        if (m > kTiny) S.big[0][0] = make_uint2(m << 16, t.z);
        else S.tiny[0] = make_uint2((m << 11) | (level0 << 17), t.z);
    }
    __syncthreads();
    auto load_box = [&](uint32_t p, float4 &l, float4 &h) {
        l = make_float4(S.box[0][p], S.box[1][p], S.box[2][p], 0.0f);
        h = make_float4(S.box[3][p], S.box[4][p], S.box[5][p], 0.0f);
    };
    uint32_t *bins = S.bins[wave];
    for (uint32_t it = 0;; ++it) {
        const uint32_t cur = it & 1u, nxt = cur ^ 1u, nbig = S.nbig[cur];
        if (nbig == 0) break;
        for (uint32_t k = wave; k < nbig; k += kWaves) {
            const uint2 task = S.big[cur][k];
            const uint32_t lo = task.x & 0xFFFFu, cnt = task.x >> 16;
            // centroid bounds and box
            uint32_t r[12];
            for (int j = 0; j < 12; ++j) r[j] = j % 6 < 3 ? 0xFFFFFFFFu : 0u;
            for (uint32_t i = lane; i < cnt; i += 64) {
                float4 l, h;
                float c[3];
                load_box(S.order[cur][lo + i], l, h);
                centroid(l, h, c);
                const float lv[3] = {l.x, l.y, l.z}, hv[3] = {h.x, h.y, h.z};
                for (int a = 0; a < 3; ++a) {
                    r[a] = min(r[a], f2ord(c[a]));
                    r[3 + a] = max(r[3 + a], f2ord(c[a]));
                    r[6 + a] = min(r[6 + a], f2ord(lv[a]));
                    r[9 + a] = max(r[9 + a], f2ord(hv[a]));
                }
            }
            for (int j = 0; j < 12; ++j) r[j] = j % 6 < 3 ? wave_min(r[j]) : wave_max(r[j]);
            float cmin[3], scale[3];
            bin_frame(r, cmin, scale);
            if (level0 + it >= kSahMedianLevel) scale[0] = scale[1] = scale[2] = 0.0f;
            SahSplit sp{-1, 0, cnt / 2};
            if (scale[0] > 0.0f || scale[1] > 0.0f || scale[2] > 0.0f) {
                clear_bins(bins, lane, 64);
                wave_lds_sync();
                for (uint32_t base = 0; base < cnt; base += 64) {
                    const bool valid = base + lane < cnt;
                    float4 l, h;
                    load_box(S.order[cur][lo + (valid ? base + lane : 0u)], l, h);
                    bin_wave(bins, valid, l, h, cmin, scale);
                }
                wave_lds_sync();
                SahSplit sz = sp;
                const uint32_t kxy = split_axes(bins, 0, scale, sp);
                const uint32_t kz = split_axes(bins, 2, scale, sz);
                if (kz < kxy) sp = sz;
                wave_lds_sync();
            }
            const uint32_t nleft = sp.nleft, id = lo0 + lo + nleft - 1u;
            // stable partition
            const float cm = sp.axis == 0 ? cmin[0] : (sp.axis == 1 ? cmin[1] : cmin[2]);
            const float sc = sp.axis == 0 ? scale[0] : (sp.axis == 1 ? scale[1] : scale[2]);
            uint32_t lrun = 0;
            for (uint32_t base = 0; base < cnt; base += 64) {
                const uint32_t i = base + lane;
                const bool valid = i < cnt;
                const uint32_t p = S.order[cur][lo + (valid ? i : 0u)];
                bool left = false;
                float4 l, h;
                load_box(p, l, h);
                if (valid) {
                    float c[3];
                    centroid(l, h, c);
                    const float ca = sp.axis == 0 ? c[0] : (sp.axis == 1 ? c[1] : c[2]);
                    left = sp.axis >= 0 ? sah_bin(ca, cm, sc) <= sp.bin : i < nleft;
                }
                const uint64_t bm = __ballot(left);
                const uint32_t lrank = lrun + (uint32_t)__popcll(bm & ((1ull << lane) - 1ull));
                if (valid) {
                    const uint32_t pos = min(left ? lrank : nleft + (i - lrank), cnt - 1u);
                    S.order[nxt][lo + pos] = (uint16_t)p;
                    if ((left ? nleft : cnt - nleft) == 1u) place_leaf(W, lo0 + lo + pos, S.gid[p], l, h);
                }
                lrun += (uint32_t)__popcll(bm);
            }
            if (lane == 0) {
                if (lrun != nleft || nleft == 0u || nleft >= cnt) atomicAdd(W.err, 1u);
                place_node(W, id, lo0 + lo, cnt, task.y, make_float4(ord2f(r[6]), ord2f(r[7]), ord2f(r[8]), 0.0f),
                           make_float4(ord2f(r[9]), ord2f(r[10]), ord2f(r[11]), 0.0f));
                for (uint32_t side = 0; side < 2; ++side) {
                    const uint32_t start = side ? lo + nleft : lo, c = side ? cnt - nleft : nleft;
                    const uint32_t link = (id << 1) | side;
                    if (c == 1u) {
                        (side ? W.right : W.left)[id] = n - 1u + lo0 + start;
                    } else if (c > kTiny) {
                        const uint32_t at = atomicAdd(&S.nbig[nxt], 1u);
                        if (at < kMaxBigs) S.big[nxt][at] = make_uint2(start | (c << 16), link);
                    } else if (c > 1u) {
                        const uint32_t at = atomicAdd(&S.ntiny, 1u);
                        if (at < kMaxTinies)
                            S.tiny[at] = make_uint2(start | (c << 11) | (nxt << 16) | ((level0 + it + 1) << 17), link);
                    }
                }
            }
        }
        __syncthreads();
        if (tid == 0) S.nbig[cur] = 0;
        __syncthreads();
        if (S.nbig[nxt] > kMaxBigs || S.ntiny > kMaxTinies || it > kSubtree) {   // block-uniform; cannot happen
            if (tid == 0) atomicAdd(W.err, 1u);
            return;
        }
    }

    // tiny nodes: group of 16 lanes, lane j = position j
    const uint32_t j = lane & 15u, g0 = lane & 48u;
    float *X = reinterpret_cast<float *>(&S.bins[0][0]) + (tid >> 4) * (9 * 16);   // [7][16] box, gid; bins; keys
    uint32_t *XU = reinterpret_cast<uint32_t *>(X);
    const uint32_t ntiny = S.ntiny;
    for (uint32_t base = wave * 4; base < ntiny; base += kWaves * 4) {
        const uint32_t k = base + (lane >> 4);
        const uint2 task = k < ntiny ? S.tiny[k] : make_uint2(0u, 0u);
        const uint32_t tlo = task.x & 0x7FFu, tcnt = (task.x >> 11) & 0x1Fu, pos0 = lo0 + tlo;
        uint32_t level = task.x >> 17;
        // this lane's primitive (by position), and its node: [slo, slo + scnt), link
        float bx[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        uint32_t gid = 0, slo = 0, scnt = j < tcnt ? tcnt : 0u, link = task.y;
        if (j < tcnt) {
            const uint32_t p = S.order[(task.x >> 16) & 1u][tlo + j];
            for (int q = 0; q < 6; ++q) bx[q] = S.box[q][p];
            gid = S.gid[p];
        }
        while (__ballot(scnt > 1u)) {
            const bool on = scnt > 1u;
            wave_lds_sync();
            for (int q = 0; q < 6; ++q) X[16 * q + j] = bx[q];
            wave_lds_sync();
            // centroid bounds of the node
            uint32_t cb[6] = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0u, 0u, 0u};
            if (on)
                for (uint32_t i = slo; i < slo + scnt; ++i)
                    for (int a = 0; a < 3; ++a) {
                        const uint32_t o = f2ord(0.5f * X[16 * a + i] + 0.5f * X[16 * (3 + a) + i]);
                        cb[a] = min(cb[a], o);
                        cb[3 + a] = max(cb[3 + a], o);
                    }
            float cmin[3], scale[3];
            bin_frame(cb, cmin, scale);
            int bin[3];
            for (int a = 0; a < 3; ++a) bin[a] = sah_bin(0.5f * bx[a] + 0.5f * bx[3 + a], cmin[a], scale[a]);
            XU[16 * 7 + j] = (uint32_t)bin[0] | ((uint32_t)bin[1] << 8) | ((uint32_t)bin[2] << 16);
            wave_lds_sync();
            // sides of the split at this lane's bin, per axis
            float ll[3][3], lh[3][3], rl[3][3], rh[3][3];
            uint32_t nl[3] = {0u, 0u, 0u};
            for (int a = 0; a < 3; ++a)
                for (int q = 0; q < 3; ++q) {
                    ll[a][q] = rl[a][q] = INFINITY;
                    lh[a][q] = rh[a][q] = -INFINITY;
                }
            if (on)
                for (uint32_t i = slo; i < slo + scnt; ++i) {
                    const uint32_t pb = XU[16 * 7 + i];
                    float b[6];
                    for (int q = 0; q < 6; ++q) b[q] = X[16 * q + i];
#pragma unroll
                    for (int a = 0; a < 3; ++a) {
                        const bool left = (int)((pb >> (8 * a)) & 0xFFu) <= bin[a];
                        nl[a] += left ? 1u : 0u;
                        for (int q = 0; q < 3; ++q) {
                            ll[a][q] = fminf(ll[a][q], left ? b[q] : INFINITY);
                            lh[a][q] = fmaxf(lh[a][q], left ? b[3 + q] : -INFINITY);
                            rl[a][q] = fminf(rl[a][q], left ? INFINITY : b[q]);
                            rh[a][q] = fmaxf(rh[a][q], left ? -INFINITY : b[3 + q]);
                        }
                    }
                }
            // this lane's best axis, then the node's best lane: least cost,
            // then axis, then bin
            uint32_t key = 0xFFFFFFFFu, ab = 0xFFFFFFFFu;
            if (on && level < kSahMedianLevel)
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    if (!(scale[a] > 0.0f) || nl[a] == 0u || nl[a] >= scnt) continue;
                    const float cost = half_area3(ll[a], lh[a]) * (float)nl[a] +
                                       half_area3(rl[a], rh[a]) * (float)(scnt - nl[a]);
                    if (!(cost < INFINITY)) continue;
                    const uint32_t o = f2ord(cost);
                    if (o < key) {
                        key = o;
                        ab = ((uint32_t)a << 8) | (uint32_t)bin[a];
                    }
                }
            XU[16 * 6 + j] = key;
            XU[16 * 8 + j] = ab;
            wave_lds_sync();
            uint32_t bk = 0xFFFFFFFFu, bab = 0xFFFFFFFFu;
            if (on)
                for (uint32_t i = slo; i < slo + scnt; ++i) {
                    const uint32_t ok = XU[16 * 6 + i], oab = XU[16 * 8 + i];
                    if (ok < bk || (ok == bk && oab < bab)) {
                        bk = ok;
                        bab = oab;
                    }
                }
            wave_lds_sync();
            bool left = false;
            if (on) {
                const uint32_t ax = bab >> 8;
                const int own = ax == 0 ? bin[0] : (ax == 1 ? bin[1] : bin[2]);
                left = bk != 0xFFFFFFFFu ? own <= (int)(bab & 0xFFu) : (j - slo) < scnt / 2u;
            }
            const uint32_t lm = (uint32_t)(__ballot(left) >> g0) & 0xFFFFu;
            if (on) {
                const uint32_t seg = ((1u << scnt) - 1u) << slo;
                const uint32_t nleft = (uint32_t)__builtin_popcount(lm & seg);
                const uint32_t lrank = (uint32_t)__builtin_popcount(lm & seg & ((1u << j) - 1u));
                const uint32_t to = left ? slo + lrank : slo + nleft + (j - slo - lrank);
                const uint32_t id = pos0 + slo + nleft - 1u;
                if (j == slo) {
                    float4 bl, bh;   // both sides of any split make the node's box
                    bl = make_float4(fminf(ll[0][0], rl[0][0]), fminf(ll[0][1], rl[0][1]), fminf(ll[0][2], rl[0][2]), 0.0f);
                    bh = make_float4(fmaxf(lh[0][0], rh[0][0]), fmaxf(lh[0][1], rh[0][1]), fmaxf(lh[0][2], rh[0][2]), 0.0f);
                    place_node(W, id, pos0 + slo, scnt, link, bl, bh);
                    if (nleft == 1u) W.left[id] = n - 1u + pos0 + slo;
                    if (scnt - nleft == 1u) W.right[id] = n - 1u + pos0 + slo + nleft;
                }
                for (int q = 0; q < 6; ++q) X[16 * q + to] = bx[q];
                XU[16 * 6 + to] = gid;
                // position j's node from here on
                const bool in_left = j < slo + nleft;
                link = (id << 1) | (in_left ? 0u : 1u);
                scnt = in_left ? nleft : scnt - nleft;
                slo = in_left ? slo : slo + nleft;
            }
            wave_lds_sync();
            if (on) {
                for (int q = 0; q < 6; ++q) bx[q] = X[16 * q + j];
                gid = XU[16 * 6 + j];
                if (scnt == 1u)
                    place_leaf(W, pos0 + j, gid, make_float4(bx[0], bx[1], bx[2], 0.0f),
                               make_float4(bx[3], bx[4], bx[5], 0.0f));
            }
            ++level;
        }
    }
}

uint64_t align256(uint64_t x) { return (x + 255) & ~255ull; }

// the work arrays inside one allocation; returns its size
uint64_t layout(uint32_t n, uint8_t *base, Work &W)
{
    const bool big = n > kSubtree;
    W.cap_tasks = big ? cap_tasks(n) : 0u;
    W.cap_chunks = big ? cap_chunks(n) : 0u;
    W.cap_small = big ? n / 2 + 1 : 1u;
    uint64_t at = 0;
    auto take = [&](uint64_t bytes) {
        uint8_t *p = base ? base + at : nullptr;
        at += align256(bytes);
        return (void *)p;
    };
    W.counts = (uint32_t *)take(kCountWords * 4);
    W.small = (uint4 *)take(W.cap_small * 16ull);
    for (int k = 0; k < 2; ++k) {
        W.tasks[k] = (uint4 *)take(W.cap_tasks * 16ull);
        W.cbounds[k] = (uint32_t *)take(W.cap_tasks * 24ull);
        W.chunks[k] = (uint2 *)take(W.cap_chunks * 8ull);
    }
    W.parts = (uint32_t *)take(W.cap_chunks * (kPartWords * 4ull));
    W.lbase = (uint32_t *)take(W.cap_chunks * 4ull);
    W.splits = (SplitRec *)take(W.cap_tasks * sizeof(SplitRec));
    W.prim[1] = (float4 *)take(big ? n * 32ull : 0ull);
    return at;
}

}  // namespace

uint64_t sah_work_bytes(uint32_t n)
{
    Work W;
    return layout(n, nullptr, W);
}

int build_binary_sah(hipStream_t s, uint32_t n, DevScratch &sc, const uint32_t *&vals_out)
{
    Work W;
    layout(n, (uint8_t *)sc.sah_work.ptr, W);
    W.prim[0] = (float4 *)sc.boxes.ptr;
    W.left = (uint32_t *)sc.left.ptr;
    W.right = (uint32_t *)sc.right.ptr;
    W.rfirst = (uint32_t *)sc.rfirst.ptr;
    W.ncount = (uint32_t *)sc.ncount.ptr;
    W.vals = (uint32_t *)sc.vals[0].ptr;
    W.wsrc = (uint32_t *)sc.wsrc.ptr;
    W.nbox = (float4 *)sc.nbox.ptr;
    W.err = (uint32_t *)sc.counters.ptr + 3;
    W.n = n;
    vals_out = W.vals;
    hipLaunchKernelGGL(k_sah_root, dim3(1), dim3(256), 0, s, W, (const uint32_t *)sc.bounds.ptr);
    uint32_t nsmall = 1;
    if (n > kSubtree) {
        // a level's tasks and chunks are counted on the device; launched blind
        // for a balanced tree's levels and three more, then as needed
        uint32_t level = 0, target = 3;
        for (uint64_t full = kSubtree; full < n; full *= 2) ++target;
        while (true) {
            for (; level < target; ++level) {
                const uint32_t tasks = level < 31 ? std::min(1u << level, W.cap_tasks) : W.cap_tasks;
                const uint32_t chunks = std::min(n / kChunk + tasks, W.cap_chunks);
                hipLaunchKernelGGL(k_sah_bin, dim3(chunks), dim3(kBinBlock), 0, s, W, level);
                hipLaunchKernelGGL(k_sah_split, dim3(tasks), dim3(kSplitBlock), 0, s, W, level);
                hipLaunchKernelGGL(k_sah_part, dim3(chunks), dim3(kBinBlock), 0, s, W, level);
            }
            SOLHIP_HIP_CHECK(hipMemcpyAsync(sc.pinned, W.counts, kCountWords * 4, hipMemcpyDeviceToHost, s));
            SOLHIP_HIP_CHECK(hipStreamSynchronize(s));
            if (sc.pinned[2 * level] == 0) break;
            target = level + 4;
            if (target >= kMaxSahLevels) {
                set_error("SAH BVH build did not converge");
                return SOLHIP_ERROR_DEVICE;
            }
        }
        nsmall = sc.pinned[kCountSmall];
        if (nsmall > W.cap_small) {
            set_error("SAH BVH build: too many subtrees");
            return SOLHIP_ERROR_DEVICE;
        }
    }
    if (nsmall) hipLaunchKernelGGL(k_sah_subtree, dim3(nsmall), dim3(kSubBlock), 0, s, W);
    SOLHIP_HIP_CHECK(hipGetLastError());
    return 0;
}

}  // namespace solhip
