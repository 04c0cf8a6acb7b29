// trace.hip -- raw ray queries (solhip_trace_rays) and small utility kernels.
#include <hip/hip_runtime.h>

#include "bvh.h"
#include "kernels.h"
#include "shading.h"
#include "traverse_step.h"

namespace solhip {

constexpr int kTraceBlock = 64;
// persistent query kernel: waves per SIMD, and idle lanes at which a wave takes
// new rays (24 instead of 16: within 2 %; 6 waves: 13 % slower at 0.4M rays, level at 2M)
#ifndef SOLHIP_TRACE_WAVES
#define SOLHIP_TRACE_WAVES 5
#endif
#ifndef SOLHIP_TRACE_REFILL
#define SOLHIP_TRACE_REFILL 16
#endif
// waves per SIMD that a small query is spread over
#ifndef SOLHIP_TRACE_SPREAD
#define SOLHIP_TRACE_SPREAD 1
#endif

// XCD-aware block order: workgroups are dispatched round-robin over the 8
// XCDs, so physical block b runs on XCD b % 8.  Mapping each XCD to a
// contiguous range of logical blocks keeps neighbouring rays (and the BVH
// nodes they touch) in one XCD's L2.
__device__ __forceinline__ uint32_t xcd_logical_block(uint32_t b, uint32_t nb)
{
    const uint32_t x = b & 7u, q = nb >> 3, r = nb & 7u;
    return x * q + min(x, r) + (b >> 3);
}

__device__ __forceinline__ void add_counts(Counters *c, const TravCounts &t, bool active)
{
    // wave-level sums, one atomic per wave and counter
    unsigned long long nodes = active ? t.nodes : 0, tris = active ? t.tris : 0, insts = active ? t.insts : 0;
    for (int off = 32; off > 0; off >>= 1) {
        nodes += __shfl_xor(nodes, off);
        tris += __shfl_xor(tris, off);
        insts += __shfl_xor(insts, off);
    }
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&c->nodes, nodes);
        atomicAdd(&c->tris, tris);
        atomicAdd(&c->insts, insts);
    }
}

// the end of a traversal kernel's wave: the launch's ray count (known without
// counting) is added once, by the first wave; one atomic per wave on that
// counter took about 15 ns each
__device__ __forceinline__ void end_wave(Counters *counters, uint32_t n, bool count, const TravCounts &tc, bool active)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&counters->rays, (unsigned long long)n);
    const uint64_t ov = __ballot(active && tc.overflow);
    if (ov && (threadIdx.x & 63) == 0) atomicAdd(&counters->overflow, (unsigned long long)__popcll(ov));
    if (count) add_counts(counters, tc, active);
}

__device__ __forceinline__ void write_hit(solhip_hit *dst, const TravState &st)
{
    const Hit h = trav_result(st);
    solhip_hit o;
    o.t = h.t;
    o.u = h.u;
    o.v = h.v;
    o.inst = h.inst;
    o.prim = h.prim;
    o.geom = h.inst == SOLHIP_MISS ? SOLHIP_MISS : 0u;
    *dst = o;
}

// One ray per lane in the first `lanes` lanes of every wave.  A query that
// would leave SIMDs without a wave is bound by the chain of steps of its slowest
// wave, and a step issues the work of all its lanes: fewer lanes per wave make
// shorter chains on SIMDs that are idle otherwise (launch_trace_rays).
template <bool ANY, bool COUNT, int MODE>
__global__ void __launch_bounds__(kTraceBlock) k_trace_rays(SceneView sv, const solhip_ray *rays, solhip_hit *hits,
                                                            uint32_t n, uint32_t lanes, Counters *counters)
{
    extern __shared__ uint2 stack[];
    const uint32_t lb = xcd_logical_block(blockIdx.x, gridDim.x);
    const uint32_t i = lb * lanes + threadIdx.x;
    const bool active = threadIdx.x < lanes && i < n;
    TravCounts tc{0, 0, 0, false};
    if (active) {
        const float4 *rp = reinterpret_cast<const float4 *>(rays + i);
        const float4 a = rp[0], b = rp[1];
        // the step traversal run to the end (trace_ray's visit order, hits
        // and counts, in fewer registers); sv.stack_depth includes its two
        // extra entries
        TravState st;
        trav_init<MODE, COUNT>(st, sv, v3(a.x, a.y, a.z), v3(b.x, b.y, b.z), a.w, b.w, 0xFFu, tc);
        while (!trav_step<ANY, COUNT, true, MODE>(st, sv, 0xFFu, stack + threadIdx.x, kTraceBlock, tc)) {
        }
        write_hit(hits + i, st);
    }
    end_wave(counters, n, COUNT, tc, active);
}

// More rays than lanes: a persistent grid whose waves take new rays for their
// idle lanes.  Rays are dealt in groups of 16: every 1024 consecutive rays go
// to the next XCD (its L2 sees whole stretches of a coherent batch), whose waves
// take groups in turn.  The deal is fixed, so no counter in memory is
// needed and overlapping launches share nothing.
template <bool ANY, bool COUNT, int MODE>
__global__ void __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(SOLHIP_TRACE_WAVES)))
k_trace_rays_persist(SceneView sv, const solhip_ray *rays, solhip_hit *hits, uint32_t n, Counters *counters)
{
    extern __shared__ uint2 stack[];
    const uint32_t lane = threadIdx.x, xcd = blockIdx.x & 7u, waves = gridDim.x >> 3, wave = blockIdx.x >> 3;
    TravCounts tc{0, 0, 0, false};
    TravState st;
    bool has = false, more = true;
    uint32_t ray = 0, taken = 0;   // rays this wave has taken so far
    while (true) {
        const uint64_t idle = __ballot(!has);
        if (more && __popcll(idle) >= SOLHIP_TRACE_REFILL) {
            const uint32_t k = taken + (uint32_t)__popcll(idle & ((1ull << lane) - 1ull));
            taken += (uint32_t)__popcll(idle);
            // the wave's k-th ray: group t of its XCD's
            const uint64_t t = wave + (uint64_t)(k >> 4) * waves;
            const uint64_t i = ((t >> 6) * 8u + xcd) * 1024u + (t & 63u) * 16u + (k & 15u);
            const bool ok = !has && i < n;
            if (ok) {
                ray = (uint32_t)i;
                const float4 *rp = reinterpret_cast<const float4 *>(rays + ray);
                const float4 a = rp[0], b = rp[1];
                trav_init<MODE, COUNT>(st, sv, v3(a.x, a.y, a.z), v3(b.x, b.y, b.z), a.w, b.w, 0xFFu, tc);
                has = true;
            }
            // groups follow one another in ray order: past the end once, past it for good
            more = __ballot(ok) == idle;
        }
        if (__ballot(has) == 0 && !more) break;
        if (has && trav_step<ANY, COUNT, true, MODE>(st, sv, 0xFFu, stack + lane, kTraceBlock, tc)) {
            write_hit(hits + ray, st);
            has = false;
        }
    }
    end_wave(counters, n, COUNT, tc, true);
}

int launch_trace_rays(hipStream_t s, const SceneView &sv, const solhip_ray *rays, solhip_hit *hits, uint32_t n,
                      uint32_t flags, uint32_t ncu, Counters *counters, Timer *timer)
{
    if (n == 0) return 0;
    if (timer) timer->begin(s, SOLHIP_KERNEL_TRACE_RAYS);
    SceneView v = sv;
    v.stack_depth += 2;
    const dim3 block(kTraceBlock);
    const size_t lds = (size_t)v.stack_depth * sizeof(uint2) * kTraceBlock;
    const bool any = flags & SOLHIP_TRACE_TERMINATE_ON_FIRST_HIT, count = flags & SOLHIP_TRACE_COUNT;
    const uint32_t simds = ncu * 4u;
    const uint32_t resident = (simds * SOLHIP_TRACE_WAVES + 7u) & ~7u;
    // Refill pays once there are more rays than lanes, except in trees of a few
    // levels, whose rays end together anyway.  Microseconds, one ray per lane
    // against refill when the rule was set: 2M rays on 131K triangles 321 / 202, on 500
    // instances 1692 / 1086 (195 and 911 since the phases are voted on), in the Cornell
    // box (6 instances of 2 to 12 triangles, depth 4) 135 / 164 (105 / - now); 0.4M rays
    // on the triangles 98.7 / 97.5.  (2M with a counter atomic per wave, as before:
    // 463, 2055 and 400.)
    if (n > resident * 64u && sv.stack_depth > kFewLevels) {
        trav_dispatch(sv.mode, count, [&](auto mode, auto cnt) {
            if constexpr (mode.value != kTravFew) {   // (a scene of that form has no more than kFewLevels)
                if (any)
                    hipLaunchKernelGGL((k_trace_rays_persist<true, cnt.value, mode.value>), dim3(resident), block, lds, s,
                                       v, rays, hits, n, counters);
                else
                    hipLaunchKernelGGL((k_trace_rays_persist<false, cnt.value, mode.value>), dim3(resident), block, lds, s,
                                       v, rays, hits, n, counters);
            }
        });
    } else {
        // lanes per wave: as many as leave a wave for every SIMD (64 rays on
        // the instances 185 -> 81 us with one ray per wave; 60,001 on the triangles 98 us with
        // full waves, 58 spread once over the SIMDs, 70 twice, 89 eight times)
        uint32_t lanes = 64;
        while (lanes > 1 && n / lanes < simds * SOLHIP_TRACE_SPREAD) lanes >>= 1;
        const dim3 grid((n + lanes - 1) / lanes);
        trav_dispatch(sv.mode, count, [&](auto mode, auto cnt) {
            if (any)
                hipLaunchKernelGGL((k_trace_rays<true, cnt.value, mode.value>), grid, block, lds, s, v, rays, hits, n,
                                   lanes, counters);
            else
                hipLaunchKernelGGL((k_trace_rays<false, cnt.value, mode.value>), grid, block, lds, s, v, rays, hits, n,
                                   lanes, counters);
        });
    }
    if (timer) timer->end(s, SOLHIP_KERNEL_TRACE_RAYS);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error(std::string("trace launch: ") + hipGetErrorString(e));
        return SOLHIP_ERROR_DEVICE;
    }
    return 0;
}

// (geometry, triangle in geometry) of hits on several-geometry BLASes: the
// geometry is the last one whose first BLAS-wide triangle is <= prim
__global__ void k_split_geometry(solhip_hit *hits, uint64_t n, const BlasRef *refs, uint32_t n_inst)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    solhip_hit h = hits[i];
    if (h.inst >= n_inst) return;   // a miss
    const uint32_t *geo = refs[h.inst].geo;
    if (!geo) return;
    uint32_t lo = 0, hi = geo[0];
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (geo[1 + mid] <= h.prim) lo = mid;
        else hi = mid;
    }
    h.prim -= geo[1 + lo];
    h.geom = lo;
    hits[i] = h;
}

int launch_split_geometry(hipStream_t s, solhip_hit *hits, uint64_t n, const BlasRef *refs, uint32_t n_inst)
{
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_split_geometry, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, s, hits, n, refs, n_inst);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error(std::string("split-geometry launch: ") + hipGetErrorString(e));
        return SOLHIP_ERROR_DEVICE;
    }
    return 0;
}

// fill kernel (used instead of hipMemsetAsync so that callers may capture
// the work into a HIP graph)
__global__ void k_fill(uint32_t *p, uint64_t n, uint32_t v)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t k = i; k < n; k += stride) p[k] = v;
}

int launch_fill(hipStream_t s, uint32_t *p, uint64_t nwords, uint32_t value)
{
    if (nwords == 0) return 0;
    uint64_t blocks = (nwords + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(k_fill, dim3((uint32_t)blocks), dim3(256), 0, s, p, nwords, value);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error(std::string("fill launch: ") + hipGetErrorString(e));
        return SOLHIP_ERROR_DEVICE;
    }
    return 0;
}

}  // namespace solhip
