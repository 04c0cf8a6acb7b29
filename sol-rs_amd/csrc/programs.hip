// programs.hip -- the ray-tracing programs as kernels.
//
//   SOLHIP_PROG_AO            plain ray-traced AO as a wavefront:
//                             k_ao_primary  generate + extend + shade of the
//                                           primary rays; hits are compacted
//                                           into the AO queue with one atomic
//                                           per block (block_append)
//                             k_ao_rays_persist  n_ao rays per queue entry, an
//                                           occlusion byte each
//                             k_ao_resolve  the bytes of a pixel into its value
//   SOLHIP_PROG_AO_GLSL       ao.rgen / ao.rchit / ao.rmiss
//   SOLHIP_PROG_PATHTRACE_GLSL pathtrace.rgen / pathtrace.rchit / pathtrace.rmiss
//   SOLHIP_PROG_DEBUG         debug.rgen / debug.rchit / debug.rmiss
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.h"
#include "shading.h"
#include "traverse.h"
#include "traverse_step.h"
#include "fetch.h"

namespace solhip {

// Waves per SIMD of the AO ray kernel: it is VALU-issue bound, so registers
// are traded against latency hiding until they spill (79 VGPRs at 6 waves; the general
// form would spill 18).  A 1080p frame, 8 rays per pixel on 2.1M triangles, frames one after
// another (2.38 ms one by one): 2582, 2370, 2280, 2559 us with 4 to 7 waves.
constexpr uint32_t ao_waves(uint32_t mode) { return mode == (uint32_t)kTravGeneral ? 5u : 6u; }
// A wave takes new rays for its idle lanes once at least this many are idle: a new ray is
// 315 instructions, an idle lane a share of every step (2297, 2280, 2304 us at 16, 20, 24).
constexpr uint32_t kAoRefill = 20;

// ---------------------------------------------------------------------------
// plain ray-traced AO (wavefront)
// ---------------------------------------------------------------------------
// the primary hit of pixel pix (ray direction d, RNG after the jitter): a hit
// becomes an AO queue entry (returns true); a miss has nothing to occlude and
// takes the value 1 at once
__device__ __forceinline__ bool ao_primary_result(const ProgArgs &A, uint32_t pix, uint32_t rng, V3 d, const Hit &h,
                                                  AoEntry &e)
{
    if (A.hits_out) store_hit(A.hits_out + pix, h);
    if (h.inst != SOLHIP_MISS) {
        const Surf sf = fetch_surface(A.tb, h.inst, h.prim, h.u, h.v);
        const float sg = sgn(dot(neg(d), sf.nrm));
        e.pixel = pix;
        e.px = sf.pos.x;
        e.py = sf.pos.y;
        e.pz = sf.pos.z;
        e.nx = sf.nrm.x * sg;
        e.ny = sf.nrm.y * sg;
        e.nz = sf.nrm.z * sg;
        e.rng = rng;
        return true;
    }
    float4 *px = A.accum + pix;
    const float4 old = *px;
    *px = make_float4(mixf(old.x, 1.0f, A.alpha), mixf(old.y, 1.0f, A.alpha), mixf(old.z, 1.0f, A.alpha), 1.0f);
    if (A.hits_out) {
        solhip_hit m;
        m.t = -1.0f;
        m.u = 0.0f;
        m.v = 0.0f;
        m.inst = SOLHIP_MISS;
        m.prim = SOLHIP_MISS;
        m.geom = SOLHIP_MISS;
        solhip_hit *dst = A.hits_out + (uint64_t)A.W * A.H + (uint64_t)pix * A.n_ao;
        for (uint32_t k = 0; k < A.n_ao; ++k) dst[k] = m;
    }
    return false;
}

// camera ray of pixel (x, y) with the jitter of ao.rgen:49-54; rng is the
// pixel's stream after the two jitter numbers
__device__ __forceinline__ void ao_camera(const ProgArgs &A, uint32_t x, uint32_t y, uint32_t &rng, V3 &o, V3 &d)
{
    rng = tea(x + y * A.W, A.frame);
    const float jx = next_rand(rng);
    const float jy = next_rand(rng);
    camera_ray(A.cam.view_inverse, A.cam.projection_inverse, x, y, A.W, A.H, jx, jy, o, d);
}

// Primary rays: one lane per pixel, a wave per 8x8 tile, kPrimaryWaves tiles per
// block, whose hits are appended to the AO queue with one atomic (1080p, 1, 2, 4
// and 8 tiles: AO frame 2.42, 2.39, 2.40, 2.42 ms; with a ray-counter atomic
// per wave beside it 2.53).  The stacks of a block are 66 KiB at kMaxStack levels.
#ifndef SOLHIP_AO_PRIMARY_WAVES
#define SOLHIP_AO_PRIMARY_WAVES 2
#endif
constexpr uint32_t kPrimaryWaves = SOLHIP_AO_PRIMARY_WAVES, kPrimaryBlock = 64 * kPrimaryWaves;

template <bool COUNT, int MODE>
__global__ void __launch_bounds__(kPrimaryBlock) k_ao_primary(ProgArgs A)
{
    extern __shared__ uint2 stack[];
    __shared__ uint32_t s_append[kPrimaryWaves + 1];
    const uint32_t tiles_x = (A.W + 7) / 8;
    const uint32_t t = xcd_block(blockIdx.x, gridDim.x) * kPrimaryWaves + (threadIdx.x >> 6);
    const uint32_t x = (t % tiles_x) * 8 + (threadIdx.x & 7), y = (t / tiles_x) * 8 + ((threadIdx.x >> 3) & 7);
    const bool active = x < A.W && y < A.H;
    TravCounts tc{0, 0, 0, false};
    bool hit = false;
    AoEntry e;
    if (active) {
        uint32_t rng;
        V3 o, d;
        ao_camera(A, x, y, rng, o, d);
        const float tmin = fmaxf(1.0f, length3(o)) * 1e-3f;
        // the step traversal run to the end: the same visit order, hits and
        // counts as trace_ray, in fewer registers
        TravState st;
        trav_init<MODE, COUNT>(st, A.sv, o, d, tmin, 10000.0f, 0xFFu, tc);
        while (!trav_step<false, COUNT, true, MODE>(st, A.sv, 0xFFu, stack + threadIdx.x, kPrimaryBlock, tc)) {
        }
        const Hit h = trav_result(st);
        hit = ao_primary_result(A, y * A.W + x, rng, d, h, e);
    }
    const uint32_t slot = block_append<kPrimaryWaves>(A.qcount, hit, s_append);
    if (hit) A.queue[slot] = e;
    count_known<COUNT>(A.counters + SOLHIP_KERNEL_AO_PRIMARY, (unsigned long long)A.W * A.H, tc);
}

// Persistent AO rays: each lane runs the resumable traversal and, when its
// ray is done, records the occlusion and (once enough lanes of the wave are
// idle) takes the next ray from a global cursor, so incoherent rays do not
// leave most of a wave waiting for its slowest lane.  Ray r = (queue entry
// r / n_ao, AO ray r % n_ao).
template <bool ANY, bool COUNT, int MODE>
__global__ void __launch_bounds__(kProgBlock) __attribute__((amdgpu_waves_per_eu(ao_waves(MODE)))) k_ao_rays_persist(ProgArgs A)
{
    extern __shared__ uint2 stack[];
    const uint32_t count = *A.qcount;
    const uint32_t total = count * A.n_ao;
    const uint32_t shift = __builtin_ctz(A.n_ao);
    const uint32_t lane = threadIdx.x & 63u;
    TravCounts tc{0, 0, 0, false};
    TravState st;
    bool has = false;
    uint32_t rid = 0, pix = 0;
    PartFetch pf;
    pf.init(A.aoheads, total);
    while (true) {
        const uint64_t idle = __ballot(!has);
        const uint32_t nidle = (uint32_t)__popcll(idle);
        if (!pf.exhausted && nidle >= kAoRefill) {
            uint32_t end;
            const uint32_t base = pf.claim(nidle, end);
            if (!has) {
                const uint32_t my = base + (uint32_t)__popcll(idle & ((1ull << lane) - 1ull));
                if (my < end) {
                    const AoEntry e = A.queue[my >> shift];
                    uint32_t rng = pcg_advance(e.rng, 2u * (my & (A.n_ao - 1u)));
                    const float xi0 = next_rand(rng);
                    const float xi1 = next_rand(rng);
                    const V3 dir = sample_cosine(v3(e.nx, e.ny, e.nz), xi0, xi1);
                    trav_init<MODE, COUNT>(st, A.sv, v3(e.px, e.py, e.pz), dir, A.ao_tmin, A.ao_tmax, 0xFFu, tc);
                    pix = e.pixel;
                    rid = my;
                    has = true;
                }
            }
        }
        if (__ballot(has) == 0 && pf.exhausted) break;
        if (has && trav_step<ANY, COUNT, true, MODE>(st, A.sv, 0xFFu, stack + threadIdx.x, kProgBlock, tc)) {
            const Hit h = trav_result(st);
            A.occl[rid] = h.inst != SOLHIP_MISS ? 1u : 0u;
            if (A.hits_out) store_hit(A.hits_out + (uint64_t)A.W * A.H + (uint64_t)pix * A.n_ao + (rid & (A.n_ao - 1u)), h);
            has = false;
        }
    }
    count_known<COUNT>(A.counters + SOLHIP_KERNEL_AO_RAYS, total, tc);
}

// one thread per queue entry: the AO value from its rays' occlusion bytes
__global__ void k_ao_resolve(ProgArgs A)
{
    const uint32_t q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= *A.qcount) return;
    const uint8_t *o = A.occl + (uint64_t)q * A.n_ao;
    uint32_t occ = 0;
    for (uint32_t k = 0; k < A.n_ao; ++k) occ += o[k];
    const float value = 1.0f - (float)occ / (float)A.n_ao;
    float4 *px = A.accum + A.queue[q].pixel;
    const float4 old = *px;
    *px = make_float4(mixf(old.x, value, A.alpha), mixf(old.y, value, A.alpha), mixf(old.z, value, A.alpha), 1.0f);
}

// dynamic LDS: the traversal stack, sv.stack_depth 8-byte entries per lane
static size_t stack_bytes(const ProgArgs &a) { return (size_t)a.sv.stack_depth * sizeof(uint2) * kProgBlock; }

static int launch_status(const char *what)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error(std::string(what) + " launch: " + hipGetErrorString(e));
        return SOLHIP_ERROR_DEVICE;
    }
    return 0;
}

#define SOLHIP_LAUNCH(kernel, id, grid, a, s, timer)                                            \
    do {                                                                                      \
        if (timer) (timer)->begin(s, id);                                                     \
        if ((a).count)                                                                        \
            hipLaunchKernelGGL(kernel<true>, dim3(grid), dim3(kProgBlock), stack_bytes(a), s, a); \
        else                                                                                  \
            hipLaunchKernelGGL(kernel<false>, dim3(grid), dim3(kProgBlock), stack_bytes(a), s, a); \
        if (timer) (timer)->end(s, id);                                                       \
    } while (0)

uint64_t ao_head_bytes() { return (uint64_t)kFetchWords * 4; }

int launch_ao(hipStream_t s, const ProgArgs &a, Timer *timer)
{
    // the step traversal (primary and persistent AO kernels) may hold two
    // more stack entries than trace_ray
    ProgArgs p = a;
    p.sv.stack_depth = a.sv.stack_depth + 2;
    const size_t lds = (size_t)p.sv.stack_depth * sizeof(uint2) * kProgBlock;
    // persistent grid: as many waves as fit on the 4 SIMDs of each CU
    const uint32_t blocks = a.ncu * 4 * ao_waves(a.sv.mode);
    // the fetch heads start at zero (a fill kernel: no memset node in a captured graph)
    int rc = launch_fill(s, a.aoheads, (uint64_t)kFetchWords, 0u);
    if (rc) return rc;
    trav_dispatch(a.sv.mode, a.count, [&](auto mode, auto count) {
        if (timer) timer->begin(s, SOLHIP_KERNEL_AO_PRIMARY);
        hipLaunchKernelGGL((k_ao_primary<count.value, mode.value>),
                           dim3((tile_count(a.W, a.H) + kPrimaryWaves - 1) / kPrimaryWaves), dim3(kPrimaryBlock),
                           lds * kPrimaryWaves, s, p);
        if (timer) timer->end(s, SOLHIP_KERNEL_AO_PRIMARY);
        if (timer) timer->begin(s, SOLHIP_KERNEL_AO_RAYS);
        if (a.ao_any)
            hipLaunchKernelGGL((k_ao_rays_persist<true, count.value, mode.value>), dim3(blocks), dim3(kProgBlock), lds, s, p);
        else
            hipLaunchKernelGGL((k_ao_rays_persist<false, count.value, mode.value>), dim3(blocks), dim3(kProgBlock), lds, s, p);
    });
    if (timer) timer->end(s, SOLHIP_KERNEL_AO_RAYS);
    const uint32_t rblocks = (a.W * a.H + kProgBlock - 1) / kProgBlock;
    hipLaunchKernelGGL(k_ao_resolve, dim3(rblocks), dim3(kProgBlock), 0, s, p);
    return launch_status("AO");
}

// ---------------------------------------------------------------------------
// The GLSL programs' pixel loops (ao.*, pathtrace.*)
// ---------------------------------------------------------------------------
// A pixel's samples follow one another (one random stream per pixel), and each
// is a chain of rays.  Two kernels run the same pixel code (AoPixel, PtPixel):
//
//   k_pixels_lockstep  one lane per pixel, each ray traced to its end before
//                      the next.  A wave waits for its slowest ray, then its longest path
//                      of every sample: cheap while paths are short.
//   k_pixels           a lane runs its pixel as a state machine on the
//                      resumable traversal: a ray that is done waits until at
//                      least SOLHIP_MEGA_SHADE lanes of the wave have something to shade, and
//                      a lane whose pixel is finished takes the block's next one.  Block b
//                      owns the 8x8 tiles b, b + grid, b + 2 grid, ... and hands out
//                      their pixels through a cursor in LDS: no device memory, so
//                      overlapping launches share nothing.
//
// Both are bound by VALU issue (0.58 wave-instructions per ns and SIMD set)
// with few lanes active.  The lockstep kernel runs the step traversal, whose
// phases a wave's lanes share whatever level of the trees they are at: with
// trace_ray's nested loops it took 1.2 (Cornell box), 1.3 (a terrain) and 2.2 times (500
// instances) as long.  Both repeat the triangle phase (trav_step's MORE) unless the
// scene is one instance: 32 bounces on the Cornell box 5.67 -> 4.9 ms, ao.* 810 ->
// 716 us; a terrain would lose 4 and 18 %.
//
// Milliseconds, lockstep against state machine, 8 samples where none are given:
//   Cornell box (kTravFew)   1280x720: depth 32 10.9 / 4.9, 8 3.5 / 3.1, 4 1.95 /
//     2.46; 500x400: depth 16 2.8 / 2.2, 8 1.52 / 1.62; 1 sample: depth 32 0.63 / 0.77;
//     300x200, 4 samples, depth 32 1.95 / 1.5; ao.*, 900x600: 0.72 / 0.89
//   terrain of 131K triangles  depth 4, 1280x720 6.2 / 4.3, 500x400 2.29 / 2.13, 1
//     sample 0.34 / 0.38, 200x150 1.51 / 1.56; ao.* 2.96 / 2.01, 1.14 / 1.04, 0.72 / 0.83
//   500 instances  depth 4, 1280x720 19.4 / 14.9, 500x400 10.7 / 9.5, 1 sample
//     1.41 / 1.57, 200x150 8.2 / 7.2; ao.* 8.1 / 6.3, 5.0 / 4.3, 3.6 / 3.5 (before the
//     instance entry's vote; with it the state machine 13.1, 8.4, lockstep 1.2, 6.8)
// waits of 16 to 64 lanes are within 4 %; 512 threads per block 5 % better than
// 256, 5 waves per SIMD spill (9.9 ms)
#ifndef SOLHIP_MEGA_SHADE
#define SOLHIP_MEGA_SHADE 48
#endif
#ifndef SOLHIP_MEGA_WAVES
#define SOLHIP_MEGA_WAVES 4
#endif
#ifndef SOLHIP_MEGA_BLOCK
#define SOLHIP_MEGA_BLOCK 512
#endif
constexpr uint32_t kMegaBlock = SOLHIP_MEGA_BLOCK;
// trav_step's MORE (scenes of one instance: 0)
constexpr int kMore = 4;

// a lane's ray
struct Segment {
    V3 o, d;
    float tmin, tmax;
};

enum class After { kRay, kSample, kPixel };   // what follows a shaded hit: another ray, a new sample, a new pixel

// ao.rgen / ao.rchit / ao.rmiss
struct AoPixel {
    static constexpr int kKernel = SOLHIP_KERNEL_AO_GLSL;
    uint32_t x, y, rng, depth;
    int sample;
    float ao, hit_value;

    __device__ __forceinline__ void begin(const ProgArgs &A, uint32_t px, uint32_t py)
    {
        x = px;
        y = py;
        ao = 0.0f;
        sample = 0;
        rng = tea(x + y * A.W, A.frame);              // ao.rgen:45
    }
    __device__ __forceinline__ void camera(const ProgArgs &A, Segment &r)
    {
        const float jx = next_rand(rng);
        const float jy = next_rand(rng);              // ao.rgen:49
        camera_ray(A.cam.view_inverse, A.cam.projection_inverse, x, y, A.W, A.H, jx, jy, r.o, r.d);
        hit_value = 0.0f;                             // preparePayload, ao.rgen:26-35
        depth = 0;
        r.tmin = fmaxf(1.0f, length3(r.o)) * 1e-3f;
        r.tmax = 10000.0f;
    }
    __device__ __forceinline__ After shade(const ProgArgs &A, const Hit &h, Segment &r)
    {
        const int max_samples = 4, sample_count = 4;  // ao.rgen:42-43
        bool done = false;
        if (h.inst == SOLHIP_MISS) {
            done = true;                              // ao.rmiss:9
        } else {
            const Surf sf = fetch_surface(A.tb, h.inst, h.prim, h.u, h.v);
            const V3 no = v3(sf.pos.x + 0.00001f * r.d.x, sf.pos.y + 0.00001f * r.d.y,
                             sf.pos.z + 0.00001f * r.d.z);   // ao.rchit:79
            const uint32_t bi = depth + depth * (uint32_t)sample;   // ao.rchit:80
            const float r0 = next_rand(rng), r1 = next_rand(rng);
            const float fw = (float)A.blue_w, fh = (float)A.blue_h;
            const float fx = (float)x + r0 * fw, fy = (float)y + r1 * fh;
            const float mx = fx - fw * floorf(fx / fw), my = fy - fh * floorf(fy / fh);
            int cx = (int)mx, cy = (int)my;
            if (cx >= (int)A.blue_w) cx -= (int)A.blue_w;
            if (cy >= (int)A.blue_h) cy -= (int)A.blue_h;
            if (cx < 0) cx += (int)A.blue_w;
            if (cy < 0) cy += (int)A.blue_h;
            const uint32_t texel = A.blue[(uint64_t)cy * A.blue_w + cx];
            const float xi0 = (float)((texel >> (8 * (bi % 4u))) & 0xFFu) / 255.0f;
            const float xi1 = (float)((texel >> (8 * ((bi + 1u) % 4u))) & 0xFFu) / 255.0f;
            const float sg = sgn(dot(neg(r.d), sf.nrm));
            const V3 hn = scale(sf.nrm, sg);                 // ao.rchit:81
            r.d = sample_cosine(hn, xi0, xi1);               // ao.rchit:82
            r.o = no;
            r.tmin = 0.001f;
            r.tmax = 10.0f;                                  // ao.rchit:83
            if (depth > 0) hit_value += 1.0f;                // ao.rchit:84-86
            depth++;
        }
        if (!done && depth <= (uint32_t)max_samples) return After::kRay;   // ao.rgen:71
        ao += 1.0f / (float)max_samples * hit_value;         // ao.rgen:74
        return ++sample < sample_count ? After::kSample : After::kPixel;
    }
    __device__ __forceinline__ void finish(const ProgArgs &A) const
    {
        const float color = 1.0f - ao / (float)4;            // ao.rgen:76
        float4 *px = A.accum + (uint64_t)y * A.W + x;
        const float4 old = *px;
        *px = make_float4(mixf(old.x, color, A.alpha), mixf(old.y, color, A.alpha), mixf(old.z, color, A.alpha), 1.0f);
    }
};

// pathtrace.rgen / pathtrace.rchit / pathtrace.rmiss
struct PtPixel {
    static constexpr int kKernel = SOLHIP_KERNEL_PATHTRACE_GLSL;
    uint32_t x, y, rng, depth;
    int sample;
    V3 pc, acc;

    __device__ __forceinline__ void begin(const ProgArgs &A, uint32_t px, uint32_t py)
    {
        x = px;
        y = py;
        sample = 0;
        pc = v3(0.0f, 0.0f, 0.0f);
        rng = tea(x + y * A.W, A.frame);   // pathtrace.rgen:47
    }
    __device__ __forceinline__ void camera(const ProgArgs &A, Segment &r)
    {
        const float jx = next_rand(rng);
        const float jy = next_rand(rng);   // :52
        camera_ray(A.cam.view_inverse, A.cam.projection_inverse, x, y, A.W, A.H, jx, jy, r.o, r.d);
        depth = 0;
        acc = v3(1.0f, 1.0f, 1.0f);
        r.tmin = fmaxf(1.0f, length3(r.o)) * 1e-3f;
        r.tmax = 10000.0f;                 // :35 (never reset)
    }
    __device__ __forceinline__ After shade(const ProgArgs &A, const Hit &h, Segment &r)
    {
        bool done = false;
        V3 hv;
        if (h.inst == SOLHIP_MISS) {
            hv = pt_miss(A.enable_sky, true, r.d);   // pathtrace.rmiss:8-21
            done = true;
        } else {
            const float *mat = reinterpret_cast<const float *>(A.tb.material_table[h.inst]);   // :69
            const float e0 = mat[4], e1 = mat[5], e2 = mat[6];
            if (e0 >= 1.0f || e1 >= 1.0f || e2 >= 1.0f) {       // :71-76
                hv = v3(e0, e1, e2);
                done = true;
                depth++;
            } else {
                const Surf sf = fetch_surface(A.tb, h.inst, h.prim, h.u, h.v);
                const V3 d = r.d;
                const V3 wI = normalize(d);                      // :90
                const float sg = sgn(dot(sf.nrm, neg(wI)));
                const V3 nO = scale(sf.nrm, sg);
                const float metallic = mat[8], roughness = mat[9];
                const float alphaSquared = roughness * roughness;
                const float xi0 = next_rand(rng);
                const float xi1 = next_rand(rng);                // :93
                const float rnd = next_rand(rng);                // :94
                r.o = v3(sf.pos.x + 0.0001f * nO.x, sf.pos.y + 0.0001f * nO.y, sf.pos.z + 0.0001f * nO.z);
                const V3 base = v3(mat[0] * sf.col.x, mat[1] * sf.col.y, mat[2] * sf.col.z);
                if (rnd < metallic) {                            // :97-100
                    r.d = sample_ggx(reflect(d, nO), xi0, xi1, alphaSquared);
                    hv = base;
                } else {
                    const V3 m = sample_ggx(nO, xi0, xi1, alphaSquared);   // :102
                    if (rnd < fresnel_dielectric(nO, m, 1.0f / 1.5f)) {
                        r.d = reflect(d, m);
                        hv = v3(1.0f, 1.0f, 1.0f);
                    } else {
                        r.d = sample_cosine(nO, xi0, xi1);
                        hv = base;
                    }
                }
                depth++;                                         // :112
            }
        }
        acc = v3(acc.x * hv.x, acc.y * hv.y, acc.z * hv.z);      // pathtrace.rgen:77
        if (!done) {
            if ((int)depth <= (int)A.max_depth) return After::kRay;
            acc = v3(0.0f, 0.0f, 0.0f);
        }
        pc = v3(pc.x + acc.x, pc.y + acc.y, pc.z + acc.z);
        return ++sample < (int)A.spp ? After::kSample : After::kPixel;
    }
    __device__ __forceinline__ void finish(const ProgArgs &A) const
    {
        const float inv = 1.0f / (float)(int)A.spp;              // :88
        float4 *px = A.accum + (uint64_t)y * A.W + x;
        const float4 old = *px;
        float m0 = mixf(old.x, inv * pc.x, A.alpha), m1 = mixf(old.y, inv * pc.y, A.alpha),
              m2 = mixf(old.z, inv * pc.z, A.alpha);
        const bool bad = isnan(m0) || isnan(m1) || isnan(m2) || isinf(m0) || isinf(m1) || isinf(m2);
        if (bad) {                                               // :94-99
            m0 = old.x;
            m1 = old.y;
            m2 = old.z;
        }
        *px = make_float4(m0, m1, m2, 1.0f);
        if (A.out_rgba8) {
            const float g = 1.0f / 2.2f;                         // :102
            const uint32_t r8 = to_unorm8(powf(m0, g)), g8 = to_unorm8(powf(m1, g)), b8 = to_unorm8(powf(m2, g));
            A.out_rgba8[(uint64_t)y * A.W + x] = r8 | (g8 << 8) | (b8 << 16) | (255u << 24);
        }
    }
};

template <class Pixel, bool COUNT, int MODE>
__global__ void __launch_bounds__(kMegaBlock) __attribute__((amdgpu_waves_per_eu(SOLHIP_MEGA_WAVES)))
k_pixels(ProgArgs A)
{
    extern __shared__ uint2 stack[];
    __shared__ uint32_t s_cursor;
    if (threadIdx.x == 0) s_cursor = 0;
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t tiles_x = (A.W + 7) >> 3, tiles = tiles_x * ((A.H + 7) >> 3);
    // pixels of this block's tiles (in 64 bits: a tile count near 2^32 times 64)
    const uint64_t items = (uint64_t)((tiles - blockIdx.x + gridDim.x - 1) / gridDim.x) * 64u;
    TravCounts tc{0, 0, 0, false};
    uint32_t rays = 0;
    TravState st;
    Pixel p;
    enum : uint32_t { kWant, kTrace, kHit, kEnd };
    uint32_t state = kWant;
    while (true) {
        const uint64_t waiting = __ballot(state == kWant || state == kHit);
        const bool tracing = __ballot(state == kTrace) != 0;
        if (!waiting && !tracing) break;
        if (!tracing || __popcll(waiting) >= SOLHIP_MEGA_SHADE) {
            Segment r;
            bool go = false, fresh = false;
            if (state == kHit) {
                r.o = st.wo;
                r.d = st.wd;
                r.tmin = st.tmin;
                r.tmax = 10000.0f;   // a pathtrace segment's; ao sets its own
                const After a = p.shade(A, trav_result(st), r);
                go = a == After::kRay;
                fresh = a == After::kSample;
                if (a == After::kPixel) {
                    p.finish(A);
                    state = kWant;
                }
            }
            // lanes without a pixel take the block's next ones
            for (uint64_t want; (want = __ballot(state == kWant)) != 0;) {
                uint32_t base = 0;
                if (lane == (uint32_t)__ffsll((unsigned long long)want) - 1u)
                    base = atomicAdd(&s_cursor, (uint32_t)__popcll(want));
                base = __shfl(base, __ffsll((unsigned long long)want) - 1);
                if (state == kWant) {
                    const uint32_t k = base + (uint32_t)__popcll(want & ((1ull << lane) - 1ull));
                    if (k >= items) {
                        state = kEnd;
                    } else {
                        const uint32_t tile = blockIdx.x + (k >> 6) * gridDim.x;
                        const uint32_t x = (tile % tiles_x) * 8 + (k & 7u), y = (tile / tiles_x) * 8 + ((k >> 3) & 7u);
                        if (x < A.W && y < A.H) {
                            p.begin(A, x, y);
                            fresh = true;
                            state = kHit;   // leaves the loop; traced below
                        }
                    }
                }
            }
            if (fresh) p.camera(A, r);
            if (go || fresh) {
                trav_init<MODE, COUNT>(st, A.sv, r.o, r.d, r.tmin, r.tmax, 0xFFu, tc);
                state = kTrace;
            }
        }
        if (state == kTrace &&
            trav_step<false, COUNT, true, MODE, MODE == kTravSingle ? 0 : kMore>(
                st, A.sv, 0xFFu, stack + threadIdx.x, (int)blockDim.x, tc)) {
            state = kHit;
            ++rays;
        }
    }
    count_rays<COUNT>(A.counters + Pixel::kKernel, rays, tc);
}

template <class Pixel, bool COUNT, int MODE>
__global__ void __launch_bounds__(kProgBlock) k_pixels_lockstep(ProgArgs A)
{
    extern __shared__ uint2 stack[];
    uint32_t x, y, rays = 0;
    TravCounts tc{0, 0, 0, false};
    if (tile_pixel(A.W, A.H, x, y)) {
        Pixel p;
        p.begin(A, x, y);
        After next = After::kSample;
        while (next != After::kPixel) {
            Segment r;
            p.camera(A, r);
            do {
                TravState st;
                trav_init<MODE, COUNT>(st, A.sv, r.o, r.d, r.tmin, r.tmax, 0xFFu, tc);
                while (!trav_step<false, COUNT, true, MODE, MODE == kTravSingle ? 0 : kMore>(
                    st, A.sv, 0xFFu, stack + threadIdx.x, kProgBlock, tc)) {
                }
                const Hit h = trav_result(st);
                ++rays;
                next = p.shade(A, h, r);
            } while (next == After::kRay);
        }
        p.finish(A);
    }
    count_rays<COUNT>(A.counters + Pixel::kKernel, rays, tc);
}

template <class Pixel>
static void launch_pixels(hipStream_t s, const ProgArgs &a)
{
    ProgArgs p = a;
    p.sv.stack_depth = a.sv.stack_depth + 2;   // the step traversal's two extra entries
    // blocks of kMegaBlock lanes, or fewer where their stacks would pass 64 KiB, so that
    // two of 512 lanes still share a CU's 160 KiB of LDS (which one workgroup may have)
    uint32_t block = kMegaBlock;
    while (block > 64 && (size_t)p.sv.stack_depth * sizeof(uint2) * block > 65536) block /= 2;
    const size_t lds = (size_t)p.sv.stack_depth * sizeof(uint2) * block;
    const uint64_t tiles = (uint64_t)((a.W + 7) / 8) * ((a.H + 7) / 8);
    const uint32_t grid = (uint32_t)std::min<uint64_t>(tiles, (uint64_t)a.ncu * (4u * SOLHIP_MEGA_WAVES * 64u / block));
    trav_dispatch(a.sv.mode, a.count, [&](auto mode, auto count) {
        hipLaunchKernelGGL((k_pixels<Pixel, count.value, mode.value>), dim3(grid), dim3(block), lds, s, p);
    });
}

template <class Pixel>
static void launch_lockstep(hipStream_t s, const ProgArgs &a)
{
    ProgArgs p = a;
    p.sv.stack_depth += 2;   // the step traversal's two extra entries
    trav_dispatch(a.sv.mode, a.count, [&](auto mode, auto count) {
        hipLaunchKernelGGL((k_pixels_lockstep<Pixel, count.value, mode.value>), dim3(tile_count(a.W, a.H)),
                           dim3(kProgBlock), stack_bytes(p), s, p);
    });
}

// Whether the state machine is the faster of the two (times above).  It evens
// out what lanes take: with a second pixel per lane (twice the resident lanes) or a
// second sample, and only where rays or paths differ enough.  In trees of a few
// levels rays hardly do, so paths must be long: 16 bounces, or 8 with a second pixel.
// Elsewhere rays do, but a small image has too few lanes to fill waves that wait.
static bool machine_pays(const ProgArgs &a, uint32_t samples, uint32_t depth)
{
    const uint64_t pixels = (uint64_t)a.W * a.H, resident = (uint64_t)a.ncu * 4u * SOLHIP_MEGA_WAVES * 64u;
    const bool refills = pixels >= 2 * resident;
    if (a.sv.mode == kTravFew) return depth >= 16 ? refills || samples >= 2 : depth >= 8 && refills;
    // long paths as before
    return refills || (samples >= 2 && (2 * pixels >= resident || depth >= 16));
}

int launch_ao_glsl(hipStream_t s, const ProgArgs &a, Timer *timer)
{
    if (timer) timer->begin(s, SOLHIP_KERNEL_AO_GLSL);
    if (machine_pays(a, 4, 5)) launch_pixels<AoPixel>(s, a);   // ao.rgen's samples and rays
    else launch_lockstep<AoPixel>(s, a);
    if (timer) timer->end(s, SOLHIP_KERNEL_AO_GLSL);
    return launch_status("AO-glsl");
}

int launch_pathtrace_glsl(hipStream_t s, const ProgArgs &a, Timer *timer)
{
    const bool machine = machine_pays(a, a.spp, a.max_depth);
    if (timer) timer->begin(s, SOLHIP_KERNEL_PATHTRACE_GLSL);
    if (machine) launch_pixels<PtPixel>(s, a);
    else launch_lockstep<PtPixel>(s, a);
    if (timer) timer->end(s, SOLHIP_KERNEL_PATHTRACE_GLSL);
    return launch_status("pathtrace");
}

// ---------------------------------------------------------------------------
// debug.rgen / debug.rchit / debug.rmiss
// ---------------------------------------------------------------------------
template <bool COUNT>
__global__ void __launch_bounds__(kProgBlock) k_debug(ProgArgs A)
{
    extern __shared__ uint2 stack[];
    uint32_t x, y;
    const bool active = tile_pixel(A.W, A.H, x, y);
    TravCounts tc{0, 0, 0, false};
    if (active) {
        V3 o, d;
        camera_ray(A.cam.view_inverse, A.cam.projection_inverse, x, y, A.W, A.H, 0.5f, 0.5f, o, d);  // debug.rgen:20-26
        const Hit h = trace_ray<false, COUNT>(A.sv, o, d, 0.001f, 1000.0f, 0xFFu, stack + threadIdx.x, kProgBlock, tc);
        float4 r;
        if (h.inst == SOLHIP_MISS)
            r = make_float4(d.x, d.y, d.z, 0.0f);                       // debug.rgen:28
        else
            r = make_float4(1.0f - h.u - h.v, h.u, h.v, 0.0f);          // debug.rchit:11-12
        A.accum[(uint64_t)y * A.W + x] = r;
    }
    count_known<COUNT>(A.counters + SOLHIP_KERNEL_DEBUG, (unsigned long long)A.W * A.H, tc);
}

int launch_debug(hipStream_t s, const ProgArgs &a, Timer *timer)
{
    const uint32_t tiles = tile_count(a.W, a.H);
    SOLHIP_LAUNCH(k_debug, SOLHIP_KERNEL_DEBUG, tiles, a, s, timer);
    return launch_status("debug");
}

}  // namespace solhip
