// bvh_build.hip -- GPU LBVH build for BLAS (triangles) and TLAS (instances).
//
// Replaces the driver's acceleration-structure build behind
// vkCmdBuildAccelerationStructuresKHR (src/ray/acceleration.rs:44-126 via
// BLAS::new 136-239 and TLAS::new/regenerate 344-467).
//
// Pipeline (all on the stream the caller passes):
//   1. primitive boxes + centroid bounds   (triangles: 3 vertex fetches at the
//      caller's stride; instances: 8 transformed corners of the BLAS root box)
//      (2 to 5 of up to kSmallTree primitives: one workgroup, k_small_tree; with
//      SOLHIP_BUILD_PREFER_FAST_TRACE bvh_sah.hip instead)
//   2. 30-bit Morton codes of the centroids (10 bits per axis)
//   3. stable LSD radix sort of (code, index), 8-bit digits: per-tile LDS
//      histograms, one exclusive scan, per-tile stable scatter whose local
//      ranks come from wave64 ballots (match on the 8 digit bits)
//   4. Karras 2012 binary radix tree (index tie-break for equal codes)
//   5. bottom-up box refit in two phases: inside each 256-leaf block with
//      LDS flags, then across blocks from the frontier nodes with one acq_rel
//      flag per node: of one workgroup up to kCrossOne leaves, agent-scope above
//   6. top-down collapse, one launch per level, to 8-wide nodes: a node
//      repeatedly opens its largest-area internal child until it has 8
//      children; children of <= leaf_max primitives become leaves, the others
//      new nodes; slots are assigned by the octant heuristic; child boxes are
//      quantised to 8 bits, rounded outward and padded by one step
//   7. leaf records in node order (48-B triangles / 64-B instances)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "bvh.h"
#include "bvh_logic.h"
#include "common.h"
#include "wave.h"

namespace solhip {

namespace {

constexpr int kBlock = 256;
constexpr int kSortItems = 8;                 // keys per thread per tile
constexpr int kSortTile = kBlock * kSortItems;  // 2048 keys

// a thread's centroid bounds, as ordered integers
struct Bounds {
    uint32_t mn[3] = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu}, mx[3] = {0u, 0u, 0u};
    __device__ __forceinline__ void add(const float lo[3], const float hi[3])
    {
        for (int a = 0; a < 3; ++a) {
            const uint32_t c = f2ord(0.5f * lo[a] + 0.5f * hi[a]);
            mn[a] = min(mn[a], c);
            mx[a] = max(mx[a], c);
        }
    }
};

// The box kernels run at most kBoxBlocks blocks: each ends with six atomics on one
// cache line, which are served one after the other (2.1M triangles: 196 us with
// a block for every 256, 72, 58, 57 with 2048, 1024, 512 blocks).
constexpr uint32_t kBoxBlocks = 1024;

// block-wide min/max of centroids, then one atomic per block and component
__device__ void reduce_bounds(const Bounds &b, uint32_t *bounds)
{
    __shared__ uint32_t smin[3][kBlock / 64], smax[3][kBlock / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        uint32_t mn = b.mn[a], mx = b.mx[a];
        for (int off = 32; off > 0; off >>= 1) {
            mn = min(mn, (uint32_t)__shfl_xor((int)mn, off));
            mx = max(mx, (uint32_t)__shfl_xor((int)mx, off));
        }
        if (lane == 0) {
            smin[a][wave] = mn;
            smax[a][wave] = mx;
        }
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        const int a = threadIdx.x;
        uint32_t mn = 0xFFFFFFFFu, mx = 0u;
        for (int w = 0; w < kBlock / 64; ++w) {
            mn = min(mn, smin[a][w]);
            mx = max(mx, smax[a][w]);
        }
        atomicMin(&bounds[a], mn);
        atomicMax(&bounds[3 + a], mx);
    }
}

__device__ __forceinline__ const GeomDesc &geom_of(const GeomDesc *geo, uint32_t n_geo, uint32_t t)
{
    return geo[geom_index(geo, n_geo, t)];
}

// vertex k of BLAS-wide triangle t of geometry G; an index value >=
// vertex_count is counted in *bad (the build then fails with an error)
__device__ __forceinline__ const float *tri_vertex(const GeomDesc &G, uint32_t t, int k, uint32_t *bad)
{
    uint32_t iv;
    if (!tri_vertex_index(G, t, k, iv)) atomicAdd(bad, 1u);
    return reinterpret_cast<const float *>(G.vbase + (uint64_t)(G.first_vertex + iv) * G.stride);
}

__global__ void __launch_bounds__(kBlock) k_tri_boxes(const GeomDesc *geo, uint32_t n_geo, uint32_t n, float4 *boxes,
                                                      uint32_t *bounds, uint32_t *bad)
{
    Bounds b;
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const GeomDesc &G = geom_of(geo, n_geo, i);
        float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
        for (int k = 0; k < 3; ++k) {
            const float *p = tri_vertex(G, i, k, bad);
            for (int a = 0; a < 3; ++a) {
                lo[a] = fminf(lo[a], p[a]);
                hi[a] = fmaxf(hi[a], p[a]);
            }
        }
        boxes[2ull * i] = make_float4(lo[0], lo[1], lo[2], __uint_as_float(i));   // its index travels with it (SAH)
        boxes[2ull * i + 1] = make_float4(hi[0], hi[1], hi[2], 0.0f);
        b.add(lo, hi);
    }
    reduce_bounds(b, bounds);
}

// instance world boxes: the 8 corners of the BLAS root box through the 3x4
// object-to-world transform, padded relatively
__global__ void __launch_bounds__(kBlock) k_inst_boxes(const solhip_instance *inst, const BlasRef *refs, uint32_t n,
                                                       float4 *boxes, uint32_t *bounds)
{
    Bounds b;
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        float lo[3], hi[3];
        instance_box(inst[i].transform, refs[i].nodes != nullptr, refs[i].root_box, lo, hi);
        boxes[2ull * i] = make_float4(lo[0], lo[1], lo[2], 0.0f);
        boxes[2ull * i + 1] = make_float4(hi[0], hi[1], hi[2], 0.0f);
        b.add(lo, hi);
    }
    reduce_bounds(b, bounds);
}

__global__ void __launch_bounds__(kBlock) k_morton(const float4 *boxes, uint32_t n, const uint32_t *bounds,
                                                   uint32_t *keys, uint32_t *vals)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const float4 lo = boxes[2ull * i], hi = boxes[2ull * i + 1];
    const float l3[3] = {lo.x, lo.y, lo.z}, h3[3] = {hi.x, hi.y, hi.z};
    const float blo[3] = {ord2f(bounds[0]), ord2f(bounds[1]), ord2f(bounds[2])};
    const float bhi[3] = {ord2f(bounds[3]), ord2f(bounds[4]), ord2f(bounds[5])};
    keys[i] = morton30(l3, h3, blo, bhi);
    vals[i] = i;
}

// ---- radix sort ---------------------------------------------------------
__global__ void __launch_bounds__(kBlock) k_hist(const uint32_t *keys, uint32_t n, int shift, uint32_t *hist,
                                                 uint32_t ntiles)
{
    __shared__ uint32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const uint64_t base = (uint64_t)blockIdx.x * kSortTile;
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        const uint64_t i = base + (uint64_t)r * kBlock + threadIdx.x;
        if (i < n) atomicAdd(&h[(keys[i] >> shift) & 0xFFu], 1u);
    }
    __syncthreads();
    hist[(uint64_t)threadIdx.x * ntiles + blockIdx.x] = h[threadIdx.x];
}

// scan of up to 1024 * kScanItems values per block; block sums out
constexpr int kScanItems = 4;
__global__ void __launch_bounds__(kBlock) k_scan_block(uint32_t *data, uint32_t n, uint32_t *block_sums)
{
    __shared__ uint32_t s[kBlock];
    const uint64_t base = (uint64_t)blockIdx.x * kBlock * kScanItems;
    uint32_t v[kScanItems];
    uint32_t sum = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const uint64_t i = base + (uint64_t)threadIdx.x * kScanItems + k;
        v[k] = i < n ? data[i] : 0u;
        sum += v[k];
    }
    s[threadIdx.x] = sum;
    __syncthreads();
    for (int off = 1; off < kBlock; off <<= 1) {
        const uint32_t t = threadIdx.x >= off ? s[threadIdx.x - off] : 0u;
        __syncthreads();
        s[threadIdx.x] += t;
        __syncthreads();
    }
    uint32_t run = s[threadIdx.x] - sum;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const uint64_t i = base + (uint64_t)threadIdx.x * kScanItems + k;
        if (i < n) data[i] = run;
        run += v[k];
    }
    if (threadIdx.x == kBlock - 1 && block_sums) block_sums[blockIdx.x] = s[kBlock - 1];
}

__global__ void __launch_bounds__(kBlock) k_scan_add(uint32_t *data, uint32_t n, const uint32_t *block_offs)
{
    const uint64_t base = (uint64_t)blockIdx.x * kBlock * kScanItems;
    const uint32_t add = block_offs[blockIdx.x];
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const uint64_t i = base + (uint64_t)threadIdx.x * kScanItems + k;
        if (i < n) data[i] += add;
    }
}

// The exclusive scan of up to kScanOne values by one workgroup: the digit counts of
// up to 64 tiles, whose scan in three launches was a third of a radix pass. 20,480
// triangles 310 -> 287 us.
constexpr uint32_t kScanOneBlock = 1024, kScanOneItems = 16, kScanOne = kScanOneBlock * kScanOneItems;
__global__ void __launch_bounds__(kScanOneBlock) k_scan_one(uint32_t *data, uint32_t n)
{
    __shared__ uint32_t wave_sum[kScanOneBlock / 64];
    const uint32_t per = (n + kScanOneBlock - 1) / kScanOneBlock, base = threadIdx.x * per;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t v[kScanOneItems], sum = 0;
#pragma unroll
    for (uint32_t k = 0; k < kScanOneItems; ++k) {
        v[k] = k < per && base + k < n ? data[base + k] : 0u;
        sum += v[k];
    }
    uint32_t incl = sum;
    for (uint32_t off = 1; off < 64; off <<= 1) {
        const uint32_t t = __shfl_up(incl, off);
        if (lane >= off) incl += t;
    }
    if (lane == 63) wave_sum[wave] = incl;
    __syncthreads();
    uint32_t run = incl - sum;
    for (uint32_t w = 0; w < wave; ++w) run += wave_sum[w];
#pragma unroll
    for (uint32_t k = 0; k < kScanOneItems; ++k) {
        if (k < per && base + k < n) data[base + k] = run;
        run += v[k];
    }
}

__global__ void __launch_bounds__(kBlock) k_scatter(const uint32_t *keys_in, const uint32_t *vals_in, uint32_t n,
                                                    int shift, const uint32_t *offs, uint32_t ntiles,
                                                    uint32_t *keys_out, uint32_t *vals_out, uint32_t *err)
{
    __shared__ uint32_t base_off[256];   // global offset of this tile's digits, advanced per round
    __shared__ uint32_t wave_cnt[kBlock / 64][256];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    base_off[threadIdx.x] = offs[(uint64_t)threadIdx.x * ntiles + blockIdx.x];
    const uint64_t tile = (uint64_t)blockIdx.x * kSortTile;
    const uint64_t lanes_below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int r = 0; r < kSortItems; ++r) {
        for (int w = 0; w < kBlock / 64; ++w) wave_cnt[w][threadIdx.x] = 0;
        __syncthreads();
        const uint64_t i = tile + (uint64_t)r * kBlock + threadIdx.x;
        const bool valid = i < n;
        const uint32_t key = valid ? keys_in[i] : 0u;
        const uint32_t val = valid ? vals_in[i] : 0u;
        const uint32_t digit = (key >> shift) & 0xFFu;
        // lanes of this wave holding the same digit (8 ballots)
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const uint64_t m = __ballot((digit >> b) & 1u);
            peers &= ((digit >> b) & 1u) ? m : ~m;
        }
        const uint32_t rank_in_wave = __popcll(peers & lanes_below);
        if (valid && rank_in_wave == 0) wave_cnt[wave][digit] = __popcll(peers);
        __syncthreads();
        if (valid) {
            uint32_t pos = base_off[digit] + rank_in_wave;
            for (int w = 0; w < wave; ++w) pos += wave_cnt[w][digit];
            if (pos < n) {
                keys_out[pos] = key;
                vals_out[pos] = val;
            } else {
                atomicAdd(err, 1u);
            }
        }
        __syncthreads();
        uint32_t tot = 0;
        for (int w = 0; w < kBlock / 64; ++w) tot += wave_cnt[w][threadIdx.x];
        base_off[threadIdx.x] += tot;
        __syncthreads();
    }
}

// ---- Karras 2012 radix tree ---------------------------------------------
__global__ void __launch_bounds__(kBlock) k_karras(const uint32_t *keys, int n, uint32_t *left, uint32_t *right,
                                                   uint32_t *parent, uint32_t *rfirst, uint32_t *ncount,
                                                   uint32_t *flags)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n - 1) return;
    karras_node(keys, n, i, left, right, parent, rfirst, ncount);
    flags[i] = 0;   // k_refit_cross's arrival flags
    if (i == 0) parent[0] = 0xFFFFFFFFu;
}

// bottom-up boxes; nbox[2*node] = lo, [2*node+1] = hi (ncount of internal
// nodes comes from k_karras: the size of the node's leaf range).
//
// Two phases.  k_refit_local: block b owns sorted leaves [256b, 256b+256);
// an internal node whose leaf range lies inside that span has its index in
// it too (one end of a radix-tree node's range is the node itself), so the
// block builds those nodes with workgroup-scope LDS flags and LDS boxes (the
// second child to arrive merges).  A node whose parent's range leaves the
// span is a frontier node: k_refit_cross walks up from the frontier nodes
// with agent-scope flags, over the few nodes that span blocks.
constexpr uint32_t kRefitSpan = kBlock;

__device__ __forceinline__ void box_union(float4 &lo, float4 &hi, float4 blo, float4 bhi)
{
    lo = make_float4(fminf(lo.x, blo.x), fminf(lo.y, blo.y), fminf(lo.z, blo.z), 0.0f);
    hi = make_float4(fmaxf(hi.x, bhi.x), fmaxf(hi.y, bhi.y), fmaxf(hi.z, bhi.z), 0.0f);
}

__global__ void __launch_bounds__(kBlock) k_refit_local(const float4 *pbox, const uint32_t *vals, int n,
                                                        const uint32_t *left, const uint32_t *right,
                                                        const uint32_t *parent, const uint32_t *rfirst,
                                                        uint32_t *ncount, float4 *nbox, uint32_t *frontier,
                                                        uint32_t *nfrontier, uint32_t *err)
{
    __shared__ uint32_t lflag[kRefitSpan];
    __shared__ float4 lbox[kRefitSpan][2];
    const uint32_t L0 = blockIdx.x * kRefitSpan, L1 = min((uint32_t)n, L0 + kRefitSpan);
    lflag[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t k = L0 + threadIdx.x;
    if (k >= L1) return;
    const uint32_t leaf_base = (uint32_t)(n - 1);
    uint32_t node = leaf_base + k;
    const uint32_t pk = vals[k];
    float4 lo = pbox[2ull * pk], hi = pbox[2ull * pk + 1];
    nbox[2ull * node] = lo;
    nbox[2ull * node + 1] = hi;
    ncount[node] = 1;
    if (n == 1) return;
    while (true) {
        const uint32_t par = parent[node];
        if (par == 0xFFFFFFFFu) break;
        if (par >= leaf_base) {
            atomicAdd(err, 1u);
            break;
        }
        const uint32_t plo = rfirst[par], phi = plo + ncount[par] - 1u;
        if (plo < L0 || phi >= L1) {
            frontier[atomicAdd(nfrontier, 1u)] = node;
            break;
        }
        const uint32_t old = __hip_atomic_fetch_add(&lflag[par - L0], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (old == 0) break;
        const uint32_t l = left[par], r = right[par];
        const uint32_t sib = l == node ? r : l;
        float4 slo, shi;
        if (sib >= leaf_base) {
            if (sib - leaf_base >= (uint32_t)n) {
                atomicAdd(err, 1u);
                break;
            }
            const uint32_t ps = vals[sib - leaf_base];
            slo = pbox[2ull * ps];
            shi = pbox[2ull * ps + 1];
        } else {
            if (sib < L0 || sib >= L1) {
                atomicAdd(err, 1u);
                break;
            }
            slo = lbox[sib - L0][0];
            shi = lbox[sib - L0][1];
        }
        box_union(lo, hi, slo, shi);
        lbox[par - L0][0] = lo;
        lbox[par - L0][1] = hi;
        nbox[2ull * par] = lo;
        nbox[2ull * par + 1] = hi;
        node = par;
    }
}

// SCOPE of the arrival flags and of the boxes behind them: up to kCrossOne leaves one
// workgroup walks the whole frontier, without the agent scope's cache writebacks at
// each of its dependent steps (builds of 14,400, 20,480, 50,000, 65,536 and 100,000 triangles
// 279, 287, 339, 372, 421 us with the GPU, 260, 265, 333, 374, 452 with one workgroup).
constexpr uint32_t kCrossOne = 32768, kCrossBlock = 1024;
template <int SCOPE>
__global__ void __launch_bounds__(kCrossBlock) k_refit_cross(int n, const uint32_t *left, const uint32_t *right,
                                                        const uint32_t *parent, uint32_t *flags, float4 *nbox,
                                                        const uint32_t *frontier, const uint32_t *nfrontier,
                                                        uint32_t *err)
{
    const uint32_t count = min(*nfrontier, (uint32_t)n);
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t f = blockIdx.x * blockDim.x + threadIdx.x; f < count; f += stride) {
        uint32_t node = frontier[f];
        float4 lo = nbox[2ull * node], hi = nbox[2ull * node + 1];
        while (true) {
            const uint32_t par = parent[node];
            if (par == 0xFFFFFFFFu) break;
            if (par >= (uint32_t)(n - 1)) {
                atomicAdd(err, 1u);
                break;
            }
            const uint32_t old = __hip_atomic_fetch_add(&flags[par], 1u, __ATOMIC_ACQ_REL, SCOPE);
            if (old == 0) break;
            const uint32_t l = left[par], r = right[par];
            if (l >= 2u * (uint32_t)n - 1u || r >= 2u * (uint32_t)n - 1u) {
                atomicAdd(err, 1u);
                break;
            }
            const uint32_t sib = l == node ? r : l;
            box_union(lo, hi, nbox[2ull * sib], nbox[2ull * sib + 1]);
            nbox[2ull * par] = lo;
            nbox[2ull * par + 1] = hi;
            node = par;
        }
    }
}

// ---- the binary tree of a small set, in one workgroup -------------------
// Codes, sort, radix tree and boxes of up to kSmallTree primitives.  The
// general path is 20 launches of a few microseconds each, whatever the size: a
// build of 12 to 1280 primitives was launches only.  A bitonic sort of (code,
// index) is the radix sort's order, the radix tree and the boxes are the same
// functions, so the tree is the same.  LDS: codes and indices while sorting,
// then codes and arrival flags; boxes of the internal nodes.  Build of
// 12 triangles 126 -> 73 us, 500 179 -> 111, 1024 198 -> 130, 2048 213 -> 157.
constexpr uint32_t kSmallTree = 2048;
constexpr uint32_t kSmallBlock = 1024;

__global__ void __launch_bounds__(kSmallBlock) k_small_tree(const float4 *pbox, uint32_t n, const uint32_t *bounds,
                                                            uint32_t *vals, uint32_t *left, uint32_t *right,
                                                            uint32_t *parent, uint32_t *rfirst, uint32_t *ncount,
                                                            float4 *nbox, uint32_t *err)
{
    __shared__ uint64_t item[kSmallTree];
    __shared__ float lbox[kSmallTree][6];
    const uint32_t tid = threadIdx.x;
    const float blo[3] = {ord2f(bounds[0]), ord2f(bounds[1]), ord2f(bounds[2])};
    const float bhi[3] = {ord2f(bounds[3]), ord2f(bounds[4]), ord2f(bounds[5])};
    uint32_t m = 1;
    while (m < n) m <<= 1;
    for (uint32_t i = tid; i < m; i += kSmallBlock) {
        uint64_t v = ~0ull;   // behind all codes (30 bits)
        if (i < n) {
            const float4 lo = pbox[2ull * i], hi = pbox[2ull * i + 1];
            const float l3[3] = {lo.x, lo.y, lo.z}, h3[3] = {hi.x, hi.y, hi.z};
            v = (uint64_t)morton30(l3, h3, blo, bhi) << 32 | i;
        }
        item[i] = v;
    }
    __syncthreads();
    for (uint32_t k = 2; k <= m; k <<= 1)
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            for (uint32_t t = tid; t < m / 2; t += kSmallBlock) {
                const uint32_t i = 2 * t - (t & (j - 1));
                const uint64_t a = item[i], b = item[i + j];
                if ((a > b) == ((i & k) == 0)) {
                    item[i] = b;
                    item[i + j] = a;
                }
            }
            __syncthreads();
        }
    uint32_t *keys = reinterpret_cast<uint32_t *>(item), *flag = keys + kSmallTree;
    const uint64_t i0 = tid < n ? item[tid] : 0ull, i1 = tid + kSmallBlock < n ? item[tid + kSmallBlock] : 0ull;
    __syncthreads();
    for (uint32_t q = 0; q < 2; ++q) {
        const uint32_t i = tid + q * kSmallBlock;
        const uint64_t v = q ? i1 : i0;
        keys[i] = (uint32_t)(v >> 32);
        flag[i] = 0;
        if (i < n) vals[i] = (uint32_t)v;
    }
    __syncthreads();
    for (uint32_t i = tid; i + 1 < n; i += kSmallBlock) karras_node(keys, (int)n, (int)i, left, right, parent, rfirst, ncount);
    if (tid == 0) parent[0] = 0xFFFFFFFFu;
    __syncthreads();
    // boxes: from each leaf upwards, the second child to arrive merges
    const uint32_t leaf_base = n - 1;
    for (uint32_t k = tid; k < n; k += kSmallBlock) {
        uint32_t node = leaf_base + k;
        const uint32_t pk = vals[k];
        float4 lo = pbox[2ull * pk], hi = pbox[2ull * pk + 1];
        nbox[2ull * node] = lo;
        nbox[2ull * node + 1] = hi;
        ncount[node] = 1;
        while (n > 1) {
            const uint32_t par = parent[node];
            if (par == 0xFFFFFFFFu) break;
            if (par >= leaf_base) {
                atomicAdd(err, 1u);
                break;
            }
            const uint32_t old = __hip_atomic_fetch_add(&flag[par], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (old == 0) break;
            const uint32_t l = left[par], rr = right[par];
            const uint32_t sib = l == node ? rr : l;
            if (sib >= leaf_base + n) {
                atomicAdd(err, 1u);
                break;
            }
            float4 slo, shi;
            if (sib >= leaf_base) {
                const uint32_t ps = vals[sib - leaf_base];
                slo = pbox[2ull * ps];
                shi = pbox[2ull * ps + 1];
            } else {
                const float *b = lbox[sib];
                slo = make_float4(b[0], b[1], b[2], 0.0f);
                shi = make_float4(b[3], b[4], b[5], 0.0f);
            }
            box_union(lo, hi, slo, shi);
            float *b = lbox[par];
            b[0] = lo.x;
            b[1] = lo.y;
            b[2] = lo.z;
            b[3] = hi.x;
            b[4] = hi.y;
            b[5] = hi.z;
            nbox[2ull * par] = lo;
            nbox[2ull * par + 1] = hi;
            node = par;
        }
    }
}

// ---- collapse to 8-wide quantised nodes ---------------------------------
// One launch per level of wide nodes, 8 lanes per node: lane c of a group
// holds child c while the node opens children, then slot c while it is
// written, so the boxes, quantised planes and leaf ranges of a node's children
// are fetched and computed side by side (bvh_logic.h's collapse_node is the
// same in one thread, whose scratch arrays and chain of ~30 dependent
// loads took 30 us for a level of one node).  Levels find their node range in device
// memory: the last workgroup of a level to finish writes the end of the next,
// so a build launches its expected number of levels without a read-back
// between them.  Node and leaf-record allocation: one 64-bit atomic per workgroup
// (both counters), after a scan over its nodes.
// k_collapse 70 -> 12 us on average; rebuilding 5 small BLASes and a
// 500-instance TLAS with 60,001 rays traced after it: 3.27 -> 1.79 ms.
constexpr int kCollapseBlock = 512;
constexpr uint32_t kCollapseNodes = kCollapseBlock / 8;
constexpr uint32_t kMaxLevels = 96;      // wide levels of a tree (a binary tree here is at most 80 deep)
// words of DevScratch::counters
constexpr uint32_t kCntTicket = 10;      // workgroups of the current level that have finished
constexpr uint32_t kCntLevels = 16;      // [kMaxLevels + 2] first node of every level
constexpr uint32_t kCntWords = kCntLevels + kMaxLevels + 2;

struct CollapseDev {
    uint32_t n, leaf_max, level;
    const uint32_t *left, *right, *rfirst, *ncount;
    const float4 *nbox;
    const uint32_t *vals;
    WideNode *wnodes;
    uint32_t *wsrc, *leaf_ids;
    uint32_t *counters;
};

__global__ void __launch_bounds__(kCollapseBlock) k_collapse(CollapseDev A)
{
    constexpr int kWaves = kCollapseBlock / 64;
    constexpr uint32_t kNone = 0xFFFFFFFFu;
    __shared__ uint4 s_node[kWaves][40];   // 8 nodes of 80 B per wave
    __shared__ uint32_t s_tot[kWaves], s_base[kWaves][2];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, c = lane & 7u, g0 = lane & 56u;
    const uint32_t n = A.n, nbin = 2u * n - 1u;
    uint32_t *levels = A.counters + kCntLevels;
    // (an allocation beyond n nodes is refused below and fails the build)
    const uint32_t begin = levels[A.level], end = min(levels[A.level + 1], n);
    // bits of a ballot that belong to this lane's group
    auto group_bits = [&](bool p) -> uint32_t { return (uint32_t)(__ballot(p) >> g0) & 0xFFu; };
    for (uint32_t base = begin + blockIdx.x * kCollapseNodes; base < end; base += gridDim.x * kCollapseNodes) {
        const uint32_t w = base + (tid >> 3);
        bool act = w < end, bad = false;
        const uint32_t b = act ? A.wsrc[w] : 0u;
        if (act && b >= nbin) {
            bad = true;
            act = false;
        }
        // lane c: child c of the node (kNone: none yet)
        uint32_t ch = kNone, cl = 0, cr = 0, cnt = 0, nc = 0;
        float4 lo = make_float4(INFINITY, INFINITY, INFINITY, 0.0f), hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.0f);
        auto fetch = [&](uint32_t id) {
            if (id >= nbin) {
                bad = true;
                ch = kNone;
                return;
            }
            ch = id;
            lo = A.nbox[2ull * id];
            hi = A.nbox[2ull * id + 1];
            cnt = A.ncount[id];
            if (id < n - 1u) {
                cl = A.left[id];
                cr = A.right[id];
            }
        };
        if (act) {
            if (b >= n - 1u) {   // single-leaf root
                nc = 1;
                if (c == 0) fetch(b);
            } else {
                nc = 2;
                if (c < 2) fetch(c ? A.right[b] : A.left[b]);
            }
        }
        // open the internal child of largest area (the first of equals) until there are 8
        for (int it = 0; it < 6; ++it) {
            const uint32_t key = ch != kNone && ch < n - 1u ? f2ord(half_area(lo, hi) + 0.0f) : 0u;
            const uint32_t m = group8_max(key);
            const uint32_t eq = group_bits(key == m);
            const uint32_t src = eq ? (uint32_t)__builtin_ctz(eq) : 0u;
            const uint32_t l = __shfl(cl, (int)(g0 + src)), r = __shfl(cr, (int)(g0 + src));
            if (m != 0u && nc < 8u) {
                if (c == src) fetch(l);
                if (c == nc) fetch(r);
                ++nc;
            }
        }
        // node box, and the child's centroid relative to its centre
        const bool has = ch != kNone;
        const float4 nlo = make_float4(group8_fmin(lo.x), group8_fmin(lo.y), group8_fmin(lo.z), 0.0f);
        const float4 nhi = make_float4(group8_fmax(hi.x), group8_fmax(hi.y), group8_fmax(hi.z), 0.0f);
        const float dx = (0.5f * lo.x + 0.5f * hi.x) - (0.5f * nlo.x + 0.5f * nhi.x);
        const float dy = (0.5f * lo.y + 0.5f * hi.y) - (0.5f * nlo.y + 0.5f * nhi.y);
        const float dz = (0.5f * lo.z + 0.5f * hi.z) - (0.5f * nlo.z + 0.5f * nhi.z);
        // octant slots: greedily the (child, slot) pair of least dot(c - p, w_s),
        // the first child, then the first slot, of equals
        uint32_t key[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const float cost = (((s & 1) ? -dx : dx) + ((s & 2) ? -dy : dy)) + ((s & 4) ? -dz : dz);
            key[s] = min(f2ord(cost + 0.0f), 0xFFFFFFFEu);
        }
        uint32_t used = 0, child_in = kNone;
        bool placed = !has;
        for (int it = 0; it < 8; ++it) {
            uint32_t bk = kNone, bs = 0;
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const bool better = !((used >> s) & 1u) && key[s] < bk;
                bk = better ? key[s] : bk;
                bs = better ? (uint32_t)s : bs;
            }
            if (placed) bk = kNone;
            const uint32_t m = group8_min(bk);
            const uint32_t eq = group_bits(bk == m);
            const uint32_t wc = eq ? (uint32_t)__builtin_ctz(eq) : 0u;
            const uint32_t ws = __shfl(bs, (int)(g0 + wc));
            if (m != kNone) {
                if (c == wc) placed = true;
                if (c == ws) child_in = wc;
                used |= 1u << ws;
            }
        }
        // lane c: slot c
        const int src = (int)(g0 + (child_in == kNone ? 0u : child_in));
        const uint32_t id = __shfl(ch, src);
        const uint32_t scnt = __shfl(cnt, src);
        const float slo[3] = {__shfl(lo.x, src), __shfl(lo.y, src), __shfl(lo.z, src)};
        const float shi[3] = {__shfl(hi.x, src), __shfl(hi.y, src), __shfl(hi.z, src)};
        const bool filled = child_in != kNone;
        const bool inner = filled && scnt > A.leaf_max, leaf = filled && !inner;
        if (group_bits(bad)) act = false;
        const uint32_t inner_slots = group_bits(inner);
        const uint32_t imask = act ? inner_slots : 0u;
        const uint32_t lcnt = act && leaf ? scnt : 0u;
        const uint32_t leaf_mask = group8(((1u << lcnt) - 1u) << (3u * c), [](uint32_t x, uint32_t y) { return x | y; });
        uint32_t poff = lcnt;
        for (int d = 1; d < 8; d <<= 1) {
            const uint32_t t = __shfl_up(poff, d, 8);
            if (c >= (uint32_t)d) poff += t;
        }
        const uint32_t nprim = __shfl(poff, (int)(g0 + 7u)), nint = (uint32_t)__builtin_popcount(imask);
        poff -= lcnt;
        // allocation: scan over the wave's nodes, then over the waves (node
        // count in the low half, leaf records in the high half)
        const uint32_t own = nint | (nprim << 16);
        uint32_t incl = own;
        for (int d = 8; d < 64; d <<= 1) {
            const uint32_t t = __shfl_up(incl, d);
            if (lane >= (uint32_t)d) incl += t;
        }
        if (lane == 63) s_tot[wave] = incl;
        __syncthreads();
        if (tid == 0) {
            uint32_t ni = 0, np = 0;
            for (int k = 0; k < kWaves; ++k) {
                s_base[k][0] = ni;
                s_base[k][1] = np;
                ni += s_tot[k] & 0xFFFFu;
                np += s_tot[k] >> 16;
            }
            unsigned long long at = 0;
            if (ni | np)
                at = atomicAdd(reinterpret_cast<unsigned long long *>(A.counters),
                               (unsigned long long)ni | ((unsigned long long)np << 32));
            for (int k = 0; k < kWaves; ++k) {
                s_base[k][0] += (uint32_t)at;
                s_base[k][1] += (uint32_t)(at >> 32);
            }
        }
        __syncthreads();
        const uint32_t child_base = nint ? s_base[wave][0] + ((incl - own) & 0xFFFFu) : 0u;
        const uint32_t prim_base = nprim ? s_base[wave][1] + ((incl - own) >> 16) : 0u;
        if ((uint64_t)child_base + nint > n || (uint64_t)prim_base + nprim > n) bad = true;
        const uint32_t first = leaf ? (id >= n - 1u ? id - (n - 1u) : A.rfirst[id]) : 0u;
        if (act && leaf && (uint64_t)first + scnt > n) bad = true;
        if (group_bits(bad)) {
            act = false;
            if (c == 0) atomicAdd(&A.counters[2], 1u);
        }
        if (act) {
            uint32_t eb[3];
            float sc[3], org[3];
            node_frame(nlo, nhi, eb, sc, org);
            uint8_t *nb = reinterpret_cast<uint8_t *>(s_node[wave]) + (lane >> 3) * kWideNodeBytes;
            for (int a = 0; a < 3; ++a) {
                int ql = 255, qh = 0;
                if (filled) quantise_range(slo[a], shi[a], org[a], sc[a], ql, qh);
                nb[32 + 8 * a + c] = (uint8_t)ql;
                nb[56 + 8 * a + c] = (uint8_t)qh;
            }
            if (c == 0) {
                uint32_t *h = reinterpret_cast<uint32_t *>(nb);
                h[0] = __float_as_uint(org[0]);
                h[1] = __float_as_uint(org[1]);
                h[2] = __float_as_uint(org[2]);
                h[3] = eb[0] | (eb[1] << 8) | (eb[2] << 16) | (imask << 24);
                h[4] = child_base;
                h[5] = prim_base;
                h[6] = leaf_mask;
                h[7] = 0u;
            }
            if (inner) A.wsrc[child_base + (uint32_t)__builtin_popcount(imask & ((1u << c) - 1u))] = id;
            if (leaf)
                for (uint32_t j = 0; j < scnt; ++j) A.leaf_ids[prim_base + poff + j] = A.vals[first + j];
        }
        // the wave's 8 nodes are 640 consecutive bytes
        const uint64_t written = __ballot(act && c == 0);
        wave_lds_sync();
        if (lane < 40u && ((written >> (8u * (lane / 5u))) & 1u))
            reinterpret_cast<uint4 *>(A.wnodes + base + wave * 8u)[lane] = s_node[wave][lane];
        wave_lds_sync();
    }
    // the last workgroup closes the level: every allocation of it has been made
    __syncthreads();
    if (tid == 0) {
        __threadfence();
        if (atomicAdd(&A.counters[kCntTicket], 1u) == gridDim.x - 1u) {
            A.counters[kCntTicket] = 0u;
            levels[A.level + 2] = atomicAdd(&A.counters[0], 0u);
        }
    }
}

// the tree is complete when the level after the `levels_run` launched ones is empty
__device__ __forceinline__ bool collapse_done(const uint32_t *counters, uint32_t levels_run)
{
    return counters[kCntLevels + levels_run] == counters[kCntLevels + levels_run + 1];
}

__global__ void __launch_bounds__(kBlock) k_write_tris(const uint32_t *leaf_ids, uint32_t n, const GeomDesc *geo,
                                                       uint32_t n_geo, TriRec *out, uint32_t *counters,
                                                       uint32_t levels_run)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n || !collapse_done(counters, levels_run)) return;
    const uint32_t p = leaf_ids[i];
    if (p >= n) {   // a failed collapse left the record unset
        atomicAdd(&counters[2], 1u);
        return;
    }
    uint32_t *bad = counters + 9;
    const GeomDesc &G = geom_of(geo, n_geo, p);
    TriRec r;
    for (int k = 0; k < 3; ++k) {
        const float *q = tri_vertex(G, p, k, bad);
        r.v[3 * k] = q[0];
        r.v[3 * k + 1] = q[1];
        r.v[3 * k + 2] = q[2];
    }
    r.prim = p;
    r.geom = (uint32_t)(&G - geo);
    r.lprim = p - G.tri_begin;
    out[i] = r;
}

__global__ void __launch_bounds__(kBlock) k_write_insts(const uint32_t *leaf_ids, uint32_t n,
                                                        const solhip_instance *inst, const BlasRef *refs,
                                                        InstRec *out, uint32_t *meta, uint32_t *counters,
                                                        uint32_t levels_run)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n || !collapse_done(counters, levels_run)) return;
    const uint32_t p = leaf_ids[i];
    if (p >= n) {   // a failed collapse left the record unset
        atomicAdd(&counters[2], 1u);
        return;
    }
    InstRec r;
    inverse3x4(inst[p].transform, r.inv);
    r.nodes = refs[p].nodes;
    r.tris = refs[p].tris;
    out[i] = r;
    meta[i] = (p & 0xFFFFFFu) | (inst[p].id_mask & 0xFF000000u);
}

// structural check of the collapsed tree before any traversal touches it, and
// the root box
__global__ void __launch_bounds__(kBlock) k_validate(const WideNode *wn, uint32_t prims, const float4 *nbox,
                                                     const uint32_t *wsrc, float *root_box, uint32_t *counters,
                                                     uint32_t levels_run)
{
    if (!collapse_done(counters, levels_run)) return;
    const uint32_t nodes = min(counters[0], prims);
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    for (uint32_t w = i; w < nodes; w += gridDim.x * kBlock)
        if (!node_valid(wn[w], w, nodes, prims)) atomicAdd(&counters[4], 1u);
    if (i == 0) {
        const uint32_t root = min(wsrc[0], 2u * prims - 2u);
        const float4 l = nbox[2ull * root], h = nbox[2ull * root + 1];
        root_box[0] = l.x;
        root_box[1] = l.y;
        root_box[2] = l.z;
        root_box[3] = h.x;
        root_box[4] = h.y;
        root_box[5] = h.z;
    }
}

// the state a build starts from: counters ([0] wide nodes allocated: the
// root), level ranges (level 0 is the root), centroid bounds, the root's
// binary node
__global__ void k_build_init(uint32_t *counters, uint32_t *bounds, uint32_t *wsrc)
{
    const uint32_t t = threadIdx.x;
    if (t < kCntWords) counters[t] = t == 0 || t == kCntLevels + 1 ? 1u : 0u;
    if (t < 6) bounds[t] = t < 3 ? 0xFFFFFFFFu : 0u;
    if (t == 0) wsrc[0] = 0u;
}

inline uint32_t cdiv(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

int exclusive_scan(hipStream_t s, uint32_t *data, uint32_t n, DevScratch &scratch, int level)
{
    const uint32_t per_block = kBlock * kScanItems;
    const uint32_t nb = cdiv(n, per_block);
    if (nb <= 1) {
        hipLaunchKernelGGL(k_scan_block, dim3(1), dim3(kBlock), 0, s, data, n, (uint32_t *)nullptr);
        return 0;
    }
    if (n <= kScanOne) {
        hipLaunchKernelGGL(k_scan_one, dim3(1), dim3(kScanOneBlock), 0, s, data, n);
        return 0;
    }
    uint32_t *sums = scratch.scan_level(level, nb);
    if (!sums) return SOLHIP_ERROR_OUT_OF_MEMORY;
    hipLaunchKernelGGL(k_scan_block, dim3(nb), dim3(kBlock), 0, s, data, n, sums);
    int rc = exclusive_scan(s, sums, nb, scratch, level + 1);
    if (rc) return rc;
    hipLaunchKernelGGL(k_scan_add, dim3(nb), dim3(kBlock), 0, s, data, n, (const uint32_t *)sums);
    return 0;
}

}  // namespace

uint32_t *DevScratch::scan_level(int level, uint32_t count)
{
    if (level >= (int)scan_bufs.size()) scan_bufs.resize(level + 1);
    DevBuf &b = scan_bufs[level];
    if (b.bytes < (uint64_t)count * 4) {
        if (b.reserve((uint64_t)count * 4) != 0) return nullptr;
    }
    return (uint32_t *)b.ptr;
}

int DevBuf::reserve(uint64_t bytes_needed)
{
    if (bytes >= bytes_needed && ptr) return 0;
    if (ptr) (void)hipFree(ptr);
    ptr = nullptr;
    bytes = 0;
    uint64_t want = std::max<uint64_t>(bytes_needed, 256);
    if (hipMalloc(&ptr, want) != hipSuccess) {
        ptr = nullptr;
        set_error("hipMalloc failed in BVH build (" + std::to_string(want) + " bytes)");
        return SOLHIP_ERROR_OUT_OF_MEMORY;
    }
    bytes = want;
    return 0;
}

void DevBuf::release()
{
    if (ptr) (void)hipFree(ptr);
    ptr = nullptr;
    bytes = 0;
}

static int build_binary_lbvh(hipStream_t s, uint32_t n, DevScratch &sc, const uint32_t *&vals_out);

// Generic build over primitive boxes already in scratch.boxes (2 float4 per
// primitive) with centroid bounds in scratch.bounds: a binary tree (Morton
// order and radix tree, or binned SAH when `sah`), then the 8-wide collapse,
// its check and the leaf records (write_leaves(levels launched)).  One
// read-back at the end, unless the tree is deeper than expected.
template <class WriteLeaves>
static int build_common(hipStream_t s, uint32_t n, uint32_t leaf_max, bool sah, DevScratch &sc, DeviceBvh &out,
                        WriteLeaves write_leaves)
{
    // counters (set by k_build_init): [0] wide nodes allocated, [1] leaf
    // records allocated, [2] collapse range errors, [3] sort / refit / SAH
    // range errors, [4] invalid nodes, [5] refit frontier size, [9] vertex
    // references out of range, kCntTicket, kCntLevels
    uint32_t *counters = (uint32_t *)sc.counters.ptr;
    uint32_t *pinned = sc.pinned;
    const uint32_t *vals = nullptr;
    if (sah) {
        int rc = build_binary_sah(s, n, sc, vals);
        if (rc) return rc;
    } else {
        int rc = build_binary_lbvh(s, n, sc, vals);
        if (rc) return rc;
    }
    CollapseDev a;
    a.n = n;
    a.leaf_max = leaf_max;
    a.left = (const uint32_t *)sc.left.ptr;
    a.right = (const uint32_t *)sc.right.ptr;
    a.rfirst = (const uint32_t *)sc.rfirst.ptr;
    a.ncount = (const uint32_t *)sc.ncount.ptr;
    a.nbox = (const float4 *)sc.nbox.ptr;
    a.vals = vals;
    a.wnodes = (WideNode *)out.nodes.ptr;
    a.wsrc = (uint32_t *)sc.wsrc.ptr;
    a.leaf_ids = (uint32_t *)sc.leaf_ids.ptr;
    a.counters = counters;
    // levels launched before the first read-back: a full 8-wide tree's and two
    // more (an empty level is a launch of a few microseconds, a read-back
    // tens of them); then three at a time
    uint32_t run = 0, target = 1;
    for (uint64_t full = 8; full < n; full *= 8) ++target;
    if (n > 8) target += 2;
    uint64_t most = 1;   // nodes the level can hold
    while (true) {
        for (; run < target; ++run) {
            a.level = run;
            const uint32_t blocks = std::min<uint32_t>(cdiv(most, kCollapseNodes), 2048u);
            hipLaunchKernelGGL(k_collapse, dim3(blocks), dim3(kCollapseBlock), 0, s, a);
            most = std::min<uint64_t>(most * 8, n);
        }
        hipLaunchKernelGGL(k_validate, dim3(std::min<uint32_t>(cdiv(n, kBlock), 2048u)), dim3(kBlock), 0, s,
                           (const WideNode *)a.wnodes, n, a.nbox, (const uint32_t *)a.wsrc, (float *)out.root_box.ptr,
                           counters, run);
        write_leaves(run);
        SOLHIP_HIP_CHECK(hipGetLastError());
        SOLHIP_HIP_CHECK(hipMemcpyAsync(pinned, counters, kCntWords * 4, hipMemcpyDeviceToHost, s));
        SOLHIP_HIP_CHECK(hipStreamSynchronize(s));
        if (pinned[9]) {
            set_error("BLAS geometry holds " + std::to_string(pinned[9]) +
                      " vertex references at or beyond its vertex_count");
            return SOLHIP_ERROR_INVALID_ARGUMENT;
        }
        if (pinned[2] || pinned[3]) {
            set_error("BVH build range check failed (collapse " + std::to_string(pinned[2]) + ", sort/refit " +
                      std::to_string(pinned[3]) + ")");
            return SOLHIP_ERROR_DEVICE;
        }
        const uint32_t *levels = pinned + kCntLevels;
        if (levels[run] == levels[run + 1]) break;
        if (levels[run + 1] > n || run + 3 > kMaxLevels) {
            set_error("BVH collapse did not converge");
            return SOLHIP_ERROR_DEVICE;
        }
        target = run + 3;
    }
    out.node_count = pinned[0];
    out.depth = 0;
    while (pinned[kCntLevels + out.depth] < pinned[kCntLevels + out.depth + 1]) ++out.depth;
    out.prim_count = n;
    if (pinned[1] != n) {
        set_error("BVH collapse placed " + std::to_string(pinned[1]) + " of " + std::to_string(n) + " primitives");
        return SOLHIP_ERROR_DEVICE;
    }
    if (pinned[4] != 0) {
        set_error("BVH validation failed on " + std::to_string(pinned[4]) + " nodes");
        return SOLHIP_ERROR_DEVICE;
    }
    return 0;
}

// Binary tree over Morton order: codes, LSD radix sort, Karras radix tree,
// two-phase refit.  Leaf order: the sorted values.
static int build_binary_lbvh(hipStream_t s, uint32_t n, DevScratch &sc, const uint32_t *&vals_out)
{
    const uint32_t g = cdiv(n, kBlock);
    uint32_t *counters = (uint32_t *)sc.counters.ptr;
    if (n <= kSmallTree) {
        hipLaunchKernelGGL(k_small_tree, dim3(1), dim3(kSmallBlock), 0, s, (const float4 *)sc.boxes.ptr, n,
                           (const uint32_t *)sc.bounds.ptr, (uint32_t *)sc.vals[0].ptr, (uint32_t *)sc.left.ptr,
                           (uint32_t *)sc.right.ptr, (uint32_t *)sc.parent.ptr, (uint32_t *)sc.rfirst.ptr,
                           (uint32_t *)sc.ncount.ptr, (float4 *)sc.nbox.ptr, counters + 3);
        vals_out = (const uint32_t *)sc.vals[0].ptr;
        return 0;
    }
    // Morton codes
    hipLaunchKernelGGL(k_morton, dim3(g), dim3(kBlock), 0, s, (const float4 *)sc.boxes.ptr, n,
                       (const uint32_t *)sc.bounds.ptr, (uint32_t *)sc.keys[0].ptr, (uint32_t *)sc.vals[0].ptr);
    // radix sort, 4 passes of 8 bits (codes have 30 bits)
    const uint32_t ntiles = cdiv(n, kSortTile);
    int cur = 0;
    for (int pass = 0; pass < 4; ++pass) {
        const int shift = pass * 8;
        hipLaunchKernelGGL(k_hist, dim3(ntiles), dim3(kBlock), 0, s, (const uint32_t *)sc.keys[cur].ptr, n, shift,
                           (uint32_t *)sc.hist.ptr, ntiles);
        int rc = exclusive_scan(s, (uint32_t *)sc.hist.ptr, 256u * ntiles, sc, 0);
        if (rc) return rc;
        hipLaunchKernelGGL(k_scatter, dim3(ntiles), dim3(kBlock), 0, s, (const uint32_t *)sc.keys[cur].ptr,
                           (const uint32_t *)sc.vals[cur].ptr, n, shift, (const uint32_t *)sc.hist.ptr, ntiles,
                           (uint32_t *)sc.keys[cur ^ 1].ptr, (uint32_t *)sc.vals[cur ^ 1].ptr, counters + 3);
        cur ^= 1;
    }
    const uint32_t *keys = (const uint32_t *)sc.keys[cur].ptr;
    const uint32_t *vals = (const uint32_t *)sc.vals[cur].ptr;
    uint32_t *left = (uint32_t *)sc.left.ptr, *right = (uint32_t *)sc.right.ptr;
    uint32_t *parent = (uint32_t *)sc.parent.ptr, *rfirst = (uint32_t *)sc.rfirst.ptr;
    uint32_t *flags = (uint32_t *)sc.flags.ptr;
    float4 *nbox = (float4 *)sc.nbox.ptr;
    uint32_t *ncount = (uint32_t *)sc.ncount.ptr;
    if (n > 1) {
        hipLaunchKernelGGL(k_karras, dim3(cdiv(n - 1, kBlock)), dim3(kBlock), 0, s, keys, (int)n, left, right, parent,
                           rfirst, ncount, flags);
    }
    uint32_t *frontier = (uint32_t *)sc.frontier.ptr;
    hipLaunchKernelGGL(k_refit_local, dim3(cdiv(n, kRefitSpan)), dim3(kBlock), 0, s, (const float4 *)sc.boxes.ptr,
                       vals, (int)n, left, right, parent, rfirst, ncount, nbox, frontier, counters + 5, counters + 3);
    if (n > 1 && n <= kCrossOne)
        hipLaunchKernelGGL(k_refit_cross<__HIP_MEMORY_SCOPE_WORKGROUP>, dim3(1), dim3(kCrossBlock), 0, s, (int)n, left,
                           right, parent, flags, nbox, frontier, counters + 5, counters + 3);
    else if (n > 1)
        hipLaunchKernelGGL(k_refit_cross<__HIP_MEMORY_SCOPE_AGENT>, dim3(std::min<uint32_t>(cdiv(n, kBlock), 2048)),
                           dim3(kBlock), 0, s, (int)n, left, right, parent, flags, nbox, frontier, counters + 5,
                           counters + 3);
    vals_out = vals;
    return 0;
}

int DevScratch::ensure(uint32_t n, bool sah)
{
    const uint64_t N = std::max<uint32_t>(n, 1);
    int rc = 0;
    rc |= boxes.reserve(N * 32);
    rc |= bounds.reserve(64);
    rc |= vals[0].reserve(N * 4);
    rc |= left.reserve(N * 4);
    rc |= right.reserve(N * 4);
    rc |= rfirst.reserve(N * 4);
    rc |= nbox.reserve(2 * N * 32);
    rc |= ncount.reserve(2 * N * 4);
    rc |= counters.reserve(kCntWords * 4);
    rc |= wsrc.reserve(N * 4);
    rc |= leaf_ids.reserve(N * 4);
    if (sah) {
        rc |= sah_work.reserve(sah_work_bytes(n));
    } else if (n <= kSmallTree) {
        rc |= parent.reserve(2 * N * 4);
    } else {
        const uint64_t ntiles = (N + kSortTile - 1) / kSortTile;
        rc |= keys[0].reserve(N * 4);
        rc |= keys[1].reserve(N * 4);
        rc |= vals[1].reserve(N * 4);
        rc |= hist.reserve(256 * ntiles * 4);
        rc |= parent.reserve(2 * N * 4);
        rc |= flags.reserve(N * 4);
        rc |= frontier.reserve(N * 4);
    }
    if (!pinned) {
        if (hipHostMalloc((void **)&pinned, kPinnedWords * 4, hipHostMallocDefault) != hipSuccess) {
            pinned = nullptr;
            set_error("hipHostMalloc failed");
            return SOLHIP_ERROR_OUT_OF_MEMORY;
        }
    }
    return rc ? SOLHIP_ERROR_OUT_OF_MEMORY : 0;
}

void DevScratch::release()
{
    for (DevBuf *b : {&boxes, &bounds, &keys[0], &keys[1], &vals[0], &vals[1], &hist, &left, &right, &parent, &rfirst,
                      &flags, &nbox, &ncount, &counters, &wsrc, &leaf_ids, &frontier, &sah_work})
        b->release();
    for (auto &b : scan_bufs) b.release();
    scan_bufs.clear();
    if (pinned) (void)hipHostFree(pinned);
    pinned = nullptr;
}

static_assert(kCntWords <= 128 && kCntWords <= kPinnedWords, "k_build_init runs one block of 128 threads");

static void launch_build_init(hipStream_t s, DevScratch &sc)
{
    hipLaunchKernelGGL(k_build_init, dim3(1), dim3(128), 0, s, (uint32_t *)sc.counters.ptr, (uint32_t *)sc.bounds.ptr,
                       (uint32_t *)sc.wsrc.ptr);
}

int build_blas(hipStream_t s, const GeomDesc *geo_dev, uint32_t n_geo, uint32_t n, uint32_t flags, DevScratch &sc,
               DeviceBvh &out)
{
    const bool sah = (flags & SOLHIP_BUILD_PREFER_FAST_TRACE) != 0 && n > 1;
    int rc = sc.ensure(n, sah);
    if (rc) return rc;
    const uint64_t nn = std::max<uint32_t>(n, 1);
    rc = out.nodes.reserve(nn * sizeof(WideNode));
    rc |= out.leaves.reserve(nn * sizeof(TriRec));
    rc |= out.root_box.reserve(64);
    if (rc) return SOLHIP_ERROR_OUT_OF_MEMORY;
    out.kind = 0;
    out.leaf_max = kLeafMaxTri;
    if (n == 0) {
        out.node_count = 0;
        out.prim_count = 0;
        out.depth = 0;
        return 0;
    }
    uint32_t *counters = (uint32_t *)sc.counters.ptr;
    launch_build_init(s, sc);
    hipLaunchKernelGGL(k_tri_boxes, dim3(std::min(cdiv(n, kBlock), kBoxBlocks)), dim3(kBlock), 0, s, geo_dev, n_geo, n,
                       (float4 *)sc.boxes.ptr, (uint32_t *)sc.bounds.ptr, counters + 9);
    return build_common(s, n, kLeafMaxTri, sah, sc, out, [&](uint32_t run) {
        hipLaunchKernelGGL(k_write_tris, dim3(cdiv(n, kBlock)), dim3(kBlock), 0, s, (const uint32_t *)sc.leaf_ids.ptr,
                           n, geo_dev, n_geo, (TriRec *)out.leaves.ptr, counters, run);
    });
}

int build_tlas(hipStream_t s, const solhip_instance *inst_dev, const BlasRef *refs_dev, uint32_t n, DevScratch &sc,
               DeviceBvh &out)
{
    int rc = sc.ensure(n, false);
    if (rc) return rc;
    const uint64_t nn = std::max<uint32_t>(n, 1);
    rc = out.nodes.reserve(nn * sizeof(WideNode));
    rc |= out.leaves.reserve(nn * sizeof(InstRec));
    rc |= out.meta.reserve(nn * 4);
    rc |= out.root_box.reserve(64);
    if (rc) return SOLHIP_ERROR_OUT_OF_MEMORY;
    out.kind = 1;
    out.leaf_max = kLeafMaxInst;
    if (n == 0) {
        out.node_count = 0;
        out.prim_count = 0;
        out.depth = 0;
        return 0;
    }
    uint32_t *counters = (uint32_t *)sc.counters.ptr;
    launch_build_init(s, sc);
    hipLaunchKernelGGL(k_inst_boxes, dim3(std::min(cdiv(n, kBlock), kBoxBlocks)), dim3(kBlock), 0, s, inst_dev, refs_dev, n,
                       (float4 *)sc.boxes.ptr, (uint32_t *)sc.bounds.ptr);
    return build_common(s, n, kLeafMaxInst, false, sc, out, [&](uint32_t run) {
        hipLaunchKernelGGL(k_write_insts, dim3(cdiv(n, kBlock)), dim3(kBlock), 0, s, (const uint32_t *)sc.leaf_ids.ptr,
                           n, inst_dev, refs_dev, (InstRec *)out.leaves.ptr, (uint32_t *)out.meta.ptr, counters, run);
    });
}

}  // namespace solhip
