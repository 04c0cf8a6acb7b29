// server.hip -- the render-request server: jobs of mixed scene, image size
// and sample count traced by one wavefront.
//
// Device state is a pool of path slots (one per pixel of every running job),
// two extension queues, a shadow queue and a list of finished slots.  One step is
//
//   trace  closest hits of every queued ray and the last step's shadow rays
//          (unoccluded contributions join the path radiance), each against its
//          job's scene
//   shade  shade_vertex (the same code as the per-frame wavefront): next ray,
//          shadow ray, or the path's sample ends.  The slot then starts its next
//          sample at once (its RNG runs on, as in pathtrace.rgen's sample loop);
//          the ended sample's radiance stays in the slot until its first shade of the next
//          step, when its last shadow ray is answered, and joins the pixel sum
//          there.  A slot without a next sample goes to the finished list: a step
//          later its pixel is accumulated into the job's image and counted done.
//
// so per pixel the arithmetic and random draws are those of the per-frame
// wavefront, in the same order: a job's image is bit-identical to a
// solhip_trace of the same program.  Admission is first-come first-served
// into free slot ranges; the trace kernel writes the per-job done counters to pinned memory,
// where the host reads a step's while the next one runs.  A run whose steps are used up
// ends by answering the last step's shadow rays and finishing its ended slots.
//
// A step of four kernels (extend, shade, shadow, retire) and a copy of the counters
// that the host waited for took 90 steps of a burst of 8 jobs 21.2 ms: 130 us of
// traversal and 25 of shading each, 55 us in retire, whose lanes counted pixels
// one atomic each on 8 addresses (15 ns apiece), 35 us between launches.  Now 13.2 ms, a
// step 110 us of trace and 28 of shade at the mean.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstring>
#include <deque>
#include <map>
#include <string>

#include "objects.h"
#include "pathshade.h"
#include "shading.h"
#include "traverse.h"
#include "traverse_step.h"
#include "fetch.h"
#include "accum.h"

namespace solhip {

namespace {

constexpr uint32_t kSrvBlock = 64;

// register budget of the trace kernel: waves per SIMD it must fit (88 to 94
// VGPRs; a burst of 8 jobs takes 13.34, 13.18, 14.7 ms with 4, 5, 6)
#ifndef SOLHIP_SRV_WAVES
#define SOLHIP_SRV_WAVES 5
#endif
#define SOLHIP_SRV_OCCUPANCY __attribute__((amdgpu_waves_per_eu(SOLHIP_SRV_WAVES)))
// words between two counters: atomics on one cache line are served one after
// the other, whichever words they meet (shade 79 us of a full step, 46 with a line each)
constexpr uint32_t kCount = 32;
constexpr uint32_t kMaxJobs = 256;   // job index lives in 8 bits of the slot meta word

// per-job constants (device array, one entry per running-job index)
struct JobDev {
    SceneView sv;
    DevTables tb;
    Cam cam;
    const LightTri *lights;
    float4 *accum;
    uint32_t *out_rgba8;
    uint32_t nlights;
    float total;
    uint32_t W, H, frame, spp, max_depth, rr_start, enable_sky, nee;
    float alpha, tmin, rmax;
    uint32_t base;      // first slot
    uint32_t streams;   // spec.sample_streams: sample s starts tea(p + s * W * H, frame)
    uint32_t lanes;     // slots per pixel (per-sample streams): slot base + j * npix + p runs samples j, j + lanes, ...
    uint32_t npix;      // W * H
};

struct SrvArgs {
    const JobDev *jobs;
    float4 *st0, *st1, *psum;
    FixSum *fsum;         // per-sample streams: per-slot order-free sums (lane 0's count: lanes done)
    uint32_t *pmeta;      // job | sample << 8
    QRay *q[2];
    QHit *hits;
    QRay *sq;
    float4 *scontrib;
    uint32_t *finished;   // max_slots words: step parity 0 fills it from the front, 1 from the back
    // counters kCount words apart, by step parity: 0, 1 extension queues, 2, 3 shadow rays, 4, 5 finished slots
    uint32_t *counts;
    uint32_t *heads;      // fetch heads of the trace kernel
    uint32_t *done;       // finished pixels per job index
    uint32_t *done_host;  // pinned: the done counters at the start of a step, by its parity
    uint32_t max_slots, max_jobs;
    uint32_t stack;       // stack entries per lane, the step traversal's two extra ones included
    Counters *counters;
};

__device__ __forceinline__ uint32_t srv_wave_append(uint32_t *counter, bool pred)
{
    const uint64_t m = __ballot(pred);
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t base = 0;
    if (m) {
        const int leader = __ffsll((unsigned long long)m) - 1;
        if ((int)lane == leader) base = atomicAdd(counter, (uint32_t)__popcll(m));
        base = __shfl(base, leader);
    }
    return base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
}

// The shade kernel runs blocks of kSrvShadeWaves waves and appends to the
// queues once per block: per-wave atomics on the few counter addresses, for
// all rays of every job, were the largest cost of a step (a burst takes 13.4, 13.4,
// 13.9 ms with 4, 8, 16 waves).
constexpr uint32_t kSrvShadeWaves = 8;
constexpr uint32_t kSrvShadeBlock = 64 * kSrvShadeWaves;

// bit of a slot's st1.w: its radiance is the ended sample's, not yet in the pixel sum
constexpr uint32_t kEnded = 0x80000000u;
constexpr uint32_t kStart = 1u << 16;   // st1.w of a new sample: depth 0, emission counts

// pathtrace.rgen:35 for this job's camera
__device__ __forceinline__ float job_tmin(const JobDev &J)
{
    float o[4];
    mat4_mul(J.cam.view_inverse, 0.0f, 0.0f, 0.0f, 1.0f, o);
    return fmaxf(1.0f, sqrtf(o[0] * o[0] + o[1] * o[1] + o[2] * o[2])) * 1e-3f;
}

// a new sample of pixel (x, y): jittered camera ray from the running RNG
__device__ __forceinline__ QRay start_sample(const JobDev &J, uint32_t slot, uint32_t x, uint32_t y, uint32_t &rng,
                                             float4 &s0, float4 &s1)
{
    const float jx = next_rand(rng);
    const float jy = next_rand(rng);
    V3 o, d;
    camera_ray(J.cam.view_inverse, J.cam.projection_inverse, x, y, J.W, J.H, jx, jy, o, d);
    s0 = make_float4(1.0f, 1.0f, 1.0f, as_f(rng));
    s1 = make_float4(0.0f, 0.0f, 0.0f, as_f(kStart));
    QRay r;
    r.ox = o.x;
    r.oy = o.y;
    r.oz = o.z;
    r.path = slot;
    r.dx = d.x;
    r.dy = d.y;
    r.dz = d.z;
    r.tmax = J.rmax;
    return r;
}

__global__ void k_srv_set_job(JobDev *jobs, uint32_t *done, uint32_t j, JobDev v)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        v.tmin = job_tmin(v);
        jobs[j] = v;
        done[j] = 0;
    }
}

// the first sample of every slot of job j (lane-major, 8x8 tiles within a
// lane), appended to queue cur; nslots = lanes * tile slots
__global__ void k_srv_admit(SrvArgs A, uint32_t j, uint32_t cur, uint32_t nslots)
{
    const JobDev &J = A.jobs[j];
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t tslots = nslots / J.lanes, ln = t / tslots, tt = t - ln * tslots;
    const uint32_t tiles_x = (J.W + 7) >> 3, tile = tt >> 6, lane = tt & 63u;
    const uint32_t x = (tile % tiles_x) * 8 + (lane & 7u), y = (tile / tiles_x) * 8 + (lane >> 3);
    const bool valid = t < nslots && x < J.W && y < J.H;
    QRay r;
    if (valid) {
        const uint32_t p = y * J.W + x, slot = J.base + ln * J.npix + p;
        // pathtrace.rgen:47; lane ln starts sample ln of its own stream
        uint32_t rng = tea(p + ln * J.npix, J.frame);
        float4 s0, s1;
        r = start_sample(J, slot, x, y, rng, s0, s1);
        A.st0[slot] = s0;
        A.st1[slot] = s1;
        if (J.streams) {
            FixSum fs;
            fix_clear(fs);
            A.fsum[slot] = fs;
        } else {
            A.psum[slot] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
        A.pmeta[slot] = j | (ln << 8);
    }
    const uint32_t at = srv_wave_append(A.counts + cur * kCount, valid);
    if (valid) A.q[cur][at] = r;
}

// One step's rays of all running jobs, each against its job's scene, through
// the resumable traversal: the extension queue, then the shadow rays that the
// last step's shading queued.  A lane takes a new ray once at least 16 lanes
// of its wave are idle.  Both kinds in one launch: a launch of either lasts as
// long as its slowest ray, and the shadow rays fill that time.  MODE: the traversal
// form that every running job's scene has, or the general one.  extend = 0: the shadow rays alone.
template <int MODE>
__global__ void __launch_bounds__(kSrvBlock) SOLHIP_SRV_OCCUPANCY k_srv_trace(SrvArgs A, uint32_t cur,
                                                                                    uint32_t extend)
{
    extern __shared__ uint2 stack[];
    const uint32_t cnt = extend ? A.counts[cur * kCount] : 0u, lane = threadIdx.x;
    const uint32_t shadows = A.counts[(2 + (cur ^ 1u)) * kCount];
    if (blockIdx.x == 0) {
        for (uint32_t j = lane; j < A.max_jobs; j += kSrvBlock) A.done_host[cur * A.max_jobs + j] = A.done[j];
        if (lane == 0) {
            // filled by this step's shading; last read a step ago
            A.counts[(cur ^ 1u) * kCount] = 0;
            A.counts[(2 + cur) * kCount] = 0;
            A.counts[(4 + cur) * kCount] = 0;
            atomicAdd(&A.counters[SOLHIP_KERNEL_SRV_EXTEND].rays, (unsigned long long)cnt);
            atomicAdd(&A.counters[SOLHIP_KERNEL_SRV_SHADOW].rays, (unsigned long long)shadows);
        }
    }
    TravCounts tc{0, 0, 0, false};
    TravState st;
    SceneView sv;
    sv.stack_depth = A.stack;
    bool has = false;
    uint32_t idx = 0, path = 0;
    PartFetch pf;
    pf.init(A.heads, cnt + shadows);
    while (true) {
        const uint64_t idle = __ballot(!has);
        const uint32_t nidle = (uint32_t)__popcll(idle);
        if (!pf.exhausted && nidle >= 16u) {
            uint32_t end;
            const uint32_t base = pf.claim(nidle, end);
            if (!has) {
                const uint32_t my = base + (uint32_t)__popcll(idle & ((1ull << lane) - 1ull));
                if (my < end) {
                    const bool any = my >= cnt;
                    idx = any ? my - cnt : my;
                    const QRay r = any ? A.sq[idx] : A.q[cur][idx];
                    const JobDev &J = A.jobs[A.pmeta[r.path] & 0xFFu];
                    sv = J.sv;
                    sv.stack_depth = A.stack;
                    trav_init<MODE, false>(st, sv, v3(r.ox, r.oy, r.oz), v3(r.dx, r.dy, r.dz), J.tmin, r.tmax, 0xFFu, tc);
                    st.any = any;
                    path = r.path;
                    has = true;
                }
            }
        }
        if (__ballot(has) == 0 && pf.exhausted) break;
        if (has &&
            trav_step<kAnyOfRay, false, true, MODE, 4>(st, sv, 0xFFu, stack + threadIdx.x, kSrvBlock, tc)) {
            const Hit h = trav_result(st);
            if (!st.any) {
                QHit out;
                out.t = h.t;
                out.u = h.u;
                out.v = h.v;
                out.inst = h.inst;
                out.prim = h.prim;
                A.hits[idx] = out;
            } else if (h.inst == SOLHIP_MISS) {
                const float4 c = A.scontrib[idx];
                float4 s1 = A.st1[path];
                s1.x = s1.x + c.x;
                s1.y = s1.y + c.y;
                s1.z = s1.z + c.z;
                A.st1[path] = s1;
            }
            has = false;
        }
    }
    count_fetches<false>(A.counters + SOLHIP_KERNEL_SRV_EXTEND, tc);
}

// the ended sample of radiance s1 joins its slot's sum
__device__ __forceinline__ void add_sample(const SrvArgs &A, const JobDev &J, uint32_t slot, float4 s1)
{
    if (J.streams) {
        FixSum fs = A.fsum[slot];
        fix_add(fs, s1.x, s1.y, s1.z);
        // field by field: lane 0's count is only ever changed atomically
        A.fsum[slot].c[0] = fs.c[0];
        A.fsum[slot].c[1] = fs.c[1];
        A.fsum[slot].c[2] = fs.c[2];
        A.fsum[slot].bad = fs.bad;
    } else {
        const float4 ps = A.psum[slot];
        A.psum[slot] = make_float4(ps.x + s1.x, ps.y + s1.y, ps.z + s1.z, 0.0f);
    }
}

// A slot's last sample has ended: it joins the sum; the pixel, once all its
// slots are there, is accumulated into the image.  True where it was.
__device__ __forceinline__ bool finish_slot(const SrvArgs &A, const JobDev &J, uint32_t slot)
{
    const uint32_t k = slot - J.base, ln = k / J.npix, p = k - ln * J.npix;
    add_sample(A, J, slot, A.st1[slot]);
    float pc0, pc1, pc2;
    bool bad = false;
    if (J.streams) {
        // this lane of the pixel is done; the pixel's last lane (counted on
        // lane 0's record) adds all of them up
        if (J.lanes > 1) {
            __threadfence();
            if (atomicAdd(&A.fsum[J.base + p].count, 1u) != J.lanes - 1u) return false;
            __threadfence();
        }
        FixSum fs = A.fsum[slot];
        for (uint32_t l = 0; l < J.lanes; ++l)
            if (l != ln) fix_merge(fs, A.fsum[J.base + l * J.npix + p]);
        pc0 = fix_value(fs.c[0]);
        pc1 = fix_value(fs.c[1]);
        pc2 = fix_value(fs.c[2]);
        bad = fs.bad;
    } else {
        const float4 ps = A.psum[slot];
        pc0 = ps.x;
        pc1 = ps.y;
        pc2 = ps.z;
    }
    // pathtrace.rgen:88-102
    const float inv = 1.0f / (float)J.spp;
    const float c0 = inv * pc0, c1 = inv * pc1, c2 = inv * pc2;
    float4 *px = J.accum + p;
    const float4 old = *px;
    float m0 = mixf(old.x, c0, J.alpha), m1 = mixf(old.y, c1, J.alpha), m2 = mixf(old.z, c2, J.alpha);
    if (bad || isnan(m0) || isnan(m1) || isnan(m2) || isinf(m0) || isinf(m1) || isinf(m2)) {
        m0 = old.x;
        m1 = old.y;
        m2 = old.z;
    }
    *px = make_float4(m0, m1, m2, 1.0f);
    if (J.out_rgba8) {
        const float g = 1.0f / 2.2f;
        const uint32_t r8 = to_unorm8(powf(m0, g)), g8 = to_unorm8(powf(m1, g)), b8 = to_unorm8(powf(m2, g));
        J.out_rgba8[p] = r8 | (g8 << 8) | (b8 << 16) | (255u << 24);
    }
    return true;
}

// Shades the queue (extend = 0: leaves it alone), then finishes the slots whose last
// sample ended a step ago.  The slots of a block that start a new sample are gathered, so that the camera code runs in
// full waves; the block appends to all its queues at once.  118 VGPRs, 4 waves per
// SIMD (a budget of 5 is 3 % slower).
__global__ void __launch_bounds__(kSrvShadeBlock) k_srv_shade(SrvArgs A, uint32_t cur, uint32_t extend)
{
    // per wave: rays that go on, shadow rays, new samples, finished slots
    __shared__ uint32_t lds[4][kSrvShadeWaves];
    __shared__ uint32_t base_of[4], again_slot[kSrvShadeBlock], again_rng[kSrvShadeBlock];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    if (blockIdx.x == 0) {
        // this step's trace is complete
        for (uint32_t k = tid; k < kFetchParts; k += blockDim.x) fetch_reset(A.heads, k);
    }
    const uint32_t cnt = extend ? A.counts[cur * kCount] : 0u;
    const uint32_t nthreads = gridDim.x * blockDim.x;
    for (uint32_t base = blockIdx.x * blockDim.x; base < cnt; base += nthreads) {
        const uint32_t i = base + tid;
        ShadeOut o;
        bool again = false, finished = false;
        uint32_t slot = 0, rng = 0;
        if (i < cnt) {
            const QRay r = A.q[cur][i];
            slot = r.path;
            const uint32_t meta = A.pmeta[slot];
            const JobDev &J = A.jobs[meta & 0xFFu];
            ShadeParams P;
            P.tb = J.tb;
            P.enable_sky = J.enable_sky;
            P.max_depth = J.max_depth;
            P.rr_start = J.rr_start;
            P.lights = J.lights;
            P.nlights = J.nlights;
            P.total = J.total;
            P.nee = J.nee && J.nlights > 0 && J.total > 0.0f;
            P.rmax = J.rmax;
            float4 s0 = A.st0[slot], s1 = A.st1[slot];
            if (as_u(s1.w) & kEnded) {
                add_sample(A, J, slot, s1);
                s1 = make_float4(0.0f, 0.0f, 0.0f, as_f(kStart));
            }
            shade_vertex(P, slot, r, A.hits[i], s0, s1, o);
            if (!o.cont) {
                const uint32_t sample = (meta >> 8) + J.lanes;   // this slot's next sample
                again = sample < J.spp;
                finished = !again;
                rng = as_u(s0.w);
                if (again) {
                    s1.w = as_f(kEnded);
                    A.pmeta[slot] = (meta & 0xFFu) | (sample << 8);
                }
            }
            if (o.cont) A.st0[slot] = s0;
            A.st1[slot] = s1;
        }
        const uint64_t below = (1ull << lane) - 1ull;
        const uint64_t m0 = __ballot(o.cont), m1 = __ballot(o.shadow), m2 = __ballot(again), m3 = __ballot(finished);
        if (lane == 0) {
            lds[0][wave] = (uint32_t)__popcll(m0);
            lds[1][wave] = (uint32_t)__popcll(m1);
            lds[2][wave] = (uint32_t)__popcll(m2);
            lds[3][wave] = (uint32_t)__popcll(m3);
        }
        __syncthreads();
        if (tid < 4) {
            uint32_t total = 0;
            for (uint32_t w = 0; w < kSrvShadeWaves; ++w) {
                const uint32_t c = lds[tid][w];
                lds[tid][w] = total;
                total += c;
            }
            // new samples stand behind the rays that go on, in the same queue
            const uint32_t news = __shfl(total, 2);
            uint32_t *counter = A.counts + (tid == 0 ? cur ^ 1u : tid == 1 ? 2 + cur : 4 + cur) * kCount;
            const uint32_t n = tid == 0 ? total + news : total;
            base_of[tid] = tid == 2 || n == 0 ? total : atomicAdd(counter, n);
        }
        __syncthreads();
        const uint32_t nagain = base_of[2];
        if (o.cont) A.q[cur ^ 1u][base_of[0] + nagain + lds[0][wave] + (uint32_t)__popcll(m0 & below)] = o.nr;
        if (o.shadow) {
            const uint32_t at = base_of[1] + lds[1][wave] + (uint32_t)__popcll(m1 & below);
            A.sq[at] = o.sr;
            A.scontrib[at] = o.sc;
        }
        if (again) {
            const uint32_t at = lds[2][wave] + (uint32_t)__popcll(m2 & below);
            again_slot[at] = slot;
            again_rng[at] = rng;
        }
        if (finished) {
            const uint32_t at = base_of[3] + lds[3][wave] + (uint32_t)__popcll(m3 & below);
            A.finished[cur ? A.max_slots - 1u - at : at] = slot;
        }
        __syncthreads();
        if (tid < nagain) {
            const uint32_t sl = again_slot[tid];
            const uint32_t meta = A.pmeta[sl];
            const JobDev &J = A.jobs[meta & 0xFFu];
            const uint32_t p = (sl - J.base) % J.npix;
            uint32_t g = J.streams ? tea(p + (meta >> 8) * J.npix, J.frame) : again_rng[tid];
            float4 s0, s1;
            const QRay r = start_sample(J, sl, p % J.W, p / J.W, g, s0, s1);
            A.st0[sl] = s0;
            A.q[cur ^ 1u][base_of[0] + tid] = r;
        }
        __syncthreads();   // LDS is reused by the next pass
    }
    const uint32_t nfin = A.counts[(4 + (cur ^ 1u)) * kCount];
    for (uint32_t base = blockIdx.x * blockDim.x; base < nfin; base += nthreads) {
        const uint32_t i = base + tid;
        uint32_t job = ~0u;
        if (i < nfin) {
            const uint32_t slot = A.finished[cur ? i : A.max_slots - 1u - i];
            const uint32_t j = A.pmeta[slot] & 0xFFu;
            if (finish_slot(A, A.jobs[j], slot)) job = j;
        }
        // finished pixels, one atomic per job and wave
        for (uint64_t left = __ballot(job != ~0u); left;) {
            const int first = __ffsll((unsigned long long)left) - 1;
            const uint64_t same = __ballot(job == (uint32_t)__shfl((int)job, first)) & left;
            if ((int)lane == first) atomicAdd(A.done + job, (uint32_t)__popcll(same));
            left &= ~same;
        }
    }
}

int srv_status(const char *what)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error(std::string(what) + " launch: " + hipGetErrorString(e));
        return SOLHIP_ERROR_DEVICE;
    }
    return 0;
}

double now_ms(std::chrono::steady_clock::time_point t0)
{
    return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
}

}  // namespace

// bytes of device state per path slot: st0, st1, psum (48), order-free sum
// (32), meta (4), two extension queues (64), hits (20), shadow queue +
// contribution (48), finished list (4)
constexpr uint64_t kSlotBytes = 48 + 32 + 4 + 64 + 20 + 48 + 4;
// slots per pixel of a job with per-sample streams when its spec leaves it
// open: enough lanes that a lane runs about kLaneSamples samples, within
// about kJobSlots slots for the job
constexpr uint32_t kLaneSamples = 16;
constexpr uint64_t kJobSlots = 4ull << 20;
constexpr uint32_t kLaneShare = 4;

struct SrvScene {
    SceneView sv;
    uint64_t tlas = 0, tlas_gen = 0;   // the TLAS and its generation at registration
    bool identity = false;             // all its instances are at the identity transform
    DevTables tb;
    DevBuf light_offsets, lights;
    uint32_t nlights = 0;
    float total = 0.0f;
};

struct SrvJob {
    solhip_job_desc desc{};
    uint32_t state = SOLHIP_JOB_QUEUED;
    double t_submit = 0, t_admit = 0, t_done = 0;
    uint32_t base = 0, npix = 0, jidx = 0;
    uint32_t lanes_max = 1;          // slots per pixel the job may use (per-sample streams)
    uint32_t lanes = 1, slots = 0;   // slots per pixel, slots of the job (lanes * npix), set at admission
    uint64_t first_step = 0;         // the first step that traces it
};

struct Server : Obj {
    Context *cx = nullptr;
    hipStream_t stream = nullptr;
    uint32_t max_slots = 0, max_jobs = 0, max_stack = 1;
    DevBuf jobs, st0, st1, psum, fsum, pmeta, q0, q1, hits, sq, scontrib, finished, counts, heads, done;
    uint32_t *done_host = nullptr;   // pinned: done counters by step parity, then those of poll()
    hipEvent_t traced[2] = {nullptr, nullptr};   // a step's trace, which writes done_host, by its parity
    std::vector<SrvScene *> scenes;
    std::map<uint64_t, SrvJob> all;
    std::deque<uint64_t> waiting;
    std::vector<uint64_t> running_by_idx;   // job id per job index (0 = free)
    std::map<uint32_t, uint32_t> free_ranges;   // start -> length
    uint64_t next_id = 1;
    uint64_t steps = 0;   // steps launched; the next one's parity is that of its queue
    std::chrono::steady_clock::time_point t0;

    SrvArgs args() const
    {
        SrvArgs a;
        std::memset(&a, 0, sizeof(a));
        a.jobs = (const JobDev *)jobs.ptr;
        a.st0 = (float4 *)st0.ptr;
        a.st1 = (float4 *)st1.ptr;
        a.psum = (float4 *)psum.ptr;
        a.fsum = (FixSum *)fsum.ptr;
        a.pmeta = (uint32_t *)pmeta.ptr;
        a.q[0] = (QRay *)q0.ptr;
        a.q[1] = (QRay *)q1.ptr;
        a.hits = (QHit *)hits.ptr;
        a.sq = (QRay *)sq.ptr;
        a.scontrib = (float4 *)scontrib.ptr;
        a.finished = (uint32_t *)finished.ptr;
        a.counts = (uint32_t *)counts.ptr;
        a.heads = (uint32_t *)heads.ptr;
        a.done = (uint32_t *)done.ptr;
        a.done_host = done_host;
        a.max_slots = max_slots;
        a.max_jobs = max_jobs;
        a.stack = max_stack + 2;   // the step traversal's two extra entries
        a.counters = cx->counters;
        return a;
    }
    bool alloc_range(uint32_t n, uint32_t &base)
    {
        for (auto it = free_ranges.begin(); it != free_ranges.end(); ++it) {
            if (it->second < n) continue;
            base = it->first;
            const uint32_t rest = it->second - n;
            free_ranges.erase(it);
            if (rest) free_ranges[base + n] = rest;
            return true;
        }
        return false;
    }
    void free_range(uint32_t base, uint32_t n)
    {
        auto it = free_ranges.emplace(base, n).first;
        auto nx = std::next(it);
        if (nx != free_ranges.end() && it->first + it->second == nx->first) {
            it->second += nx->second;
            free_ranges.erase(nx);
        }
        if (it != free_ranges.begin()) {
            auto pv = std::prev(it);
            if (pv->first + pv->second == it->first) {
                pv->second += it->second;
                free_ranges.erase(it);
            }
        }
    }
    void release_all()
    {
        for (DevBuf *b : {&jobs, &st0, &st1, &psum, &fsum, &pmeta, &q0, &q1, &hits, &sq, &scontrib, &finished, &counts, &heads,
                          &done})
            b->release();
        for (SrvScene *sc : scenes) {
            sc->light_offsets.release();
            sc->lights.release();
            delete sc;
        }
        scenes.clear();
        if (done_host) (void)hipHostFree(done_host);
        done_host = nullptr;
        for (hipEvent_t &e : traced) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
        if (stream) (void)hipStreamDestroy(stream);
        stream = nullptr;
    }

    // admit waiting jobs (first come, first served) while slots and job
    // indices are free
    int admit()
    {
        while (!waiting.empty()) {
            SrvJob &jb = all[waiting.front()];
            uint32_t jidx = 0;
            while (jidx < max_jobs && running_by_idx[jidx]) ++jidx;
            if (jidx == max_jobs) return 0;
            // slots per pixel: what the job asks for, but extra lanes take at
            // most 1/kLaneShare of the largest free range, so that jobs
            // behind it are not kept waiting; one lane if that is all that fits
            uint64_t lanes = jb.lanes_max, largest = 0;
            for (const auto &r : free_ranges) largest = std::max<uint64_t>(largest, r.second);
            lanes = std::max<uint64_t>(1, std::min<uint64_t>(lanes, largest / ((uint64_t)kLaneShare * jb.npix)));
            uint32_t base = 0;
            if (!alloc_range((uint32_t)(lanes * jb.npix), base)) {
                if (lanes == 1 || !alloc_range(jb.npix, base)) return 0;
                lanes = 1;
            }
            jb.lanes = (uint32_t)lanes;
            jb.slots = jb.lanes * jb.npix;
            const SrvScene *sc = scenes[jb.desc.scene];
            Buffer *acc = get<Buffer>(jb.desc.accum, Kind::Buffer);
            Buffer *out = jb.desc.out_rgba8 ? get<Buffer>(jb.desc.out_rgba8, Kind::Buffer) : nullptr;
            if (!acc) {
                free_range(base, jb.slots);
                return bad_handle("job accum buffer");
            }
            JobDev v;
            std::memset(&v, 0, sizeof(v));
            v.sv = sc->sv;
            v.tb = sc->tb;
            std::memcpy(v.cam.view_inverse, jb.desc.uniforms.view_inverse, 64);
            std::memcpy(v.cam.projection_inverse, jb.desc.uniforms.projection_inverse, 64);
            v.lights = (const LightTri *)sc->lights.ptr;
            v.nlights = sc->nlights;
            v.total = sc->total;
            v.accum = (float4 *)acc->ptr;
            v.out_rgba8 = out ? (uint32_t *)out->ptr : nullptr;
            v.W = jb.desc.W;
            v.H = jb.desc.H;
            v.frame = jb.desc.uniforms.frame[2];
            v.spp = jb.desc.spec.spp_per_frame;
            v.max_depth = jb.desc.spec.max_depth;
            v.rr_start = jb.desc.spec.rr_start;
            v.enable_sky = jb.desc.spec.enable_sky;
            v.nee = jb.desc.spec.nee;
            v.streams = jb.desc.spec.sample_streams;
            const uint32_t denom = jb.desc.uniforms.frame[2] - (uint32_t)jb.desc.accum_start_frame + 1u;
            v.alpha = 1.0f / (float)denom;   // pathtrace.rgen:90
            v.rmax = 10000.0f;
            v.base = base;
            v.lanes = jb.lanes;
            v.npix = jb.npix;
            hipLaunchKernelGGL(k_srv_set_job, dim3(1), dim3(64), 0, stream, (JobDev *)jobs.ptr, (uint32_t *)done.ptr,
                               jidx, v);
            const uint32_t tiles = ((v.W + 7) / 8) * ((v.H + 7) / 8), nslots = tiles * 64 * jb.lanes;
            Timer *timer = cx->timer_or_null();
            if (timer) timer->begin(stream, SOLHIP_KERNEL_SRV_ADMIT);
            hipLaunchKernelGGL(k_srv_admit, dim3((nslots + kSrvBlock - 1) / kSrvBlock), dim3(kSrvBlock), 0, stream,
                               args(), jidx, (uint32_t)(steps & 1u), nslots);
            if (timer) timer->end(stream, SOLHIP_KERNEL_SRV_ADMIT);
            int rc = srv_status("server admit");
            if (rc) return rc;
            jb.state = SOLHIP_JOB_RUNNING;
            jb.base = base;
            jb.jidx = jidx;
            jb.t_admit = now_ms(t0);
            jb.first_step = steps;
            running_by_idx[jidx] = waiting.front();
            waiting.pop_front();
        }
        return 0;
    }

    // slots of the running jobs, and a traversal form that all their scenes have:
    // one instance at the identity transform can be traversed either way
    void running(uint64_t &slots, uint32_t &mode)
    {
        bool single = true, identity = true;
        slots = 0;
        for (uint64_t id : running_by_idx) {
            if (!id) continue;
            const SrvJob &jb = all[id];
            const SrvScene *sc = scenes[jb.desc.scene];
            slots += jb.slots;
            single = single && sc->sv.mode == kTravSingle;
            identity = identity && sc->identity;
        }
        mode = single ? kTravSingle : identity ? kTravIdentity : kTravGeneral;
    }

    // a step's two kernels on the queue of parity cur
    int launch(uint32_t cur, uint32_t extend)
    {
        const SrvArgs a = args();
        uint64_t slots;
        uint32_t mode;
        running(slots, mode);
        // every slot has at most one extension and one shadow ray
        const uint32_t trace_blocks = (uint32_t)std::min<uint64_t>(cx->ncu * 4 * SOLHIP_SRV_WAVES, (2 * slots + 63) / 64);
        const uint32_t shade_blocks =
            (uint32_t)std::min<uint64_t>((slots + kSrvShadeBlock - 1) / kSrvShadeBlock, cx->ncu * 32 / kSrvShadeWaves);
        const size_t lds = (size_t)a.stack * sizeof(uint2) * kSrvBlock;
        Timer *timer = cx->timer_or_null();
        auto timed = [&](int id, auto &&launch) {
            if (timer) timer->begin(stream, id);
            launch();
            if (timer) timer->end(stream, id);
        };
        timed(SOLHIP_KERNEL_SRV_EXTEND, [&] {
            auto go = [&](auto m) {
                hipLaunchKernelGGL((k_srv_trace<m.value>), dim3(trace_blocks), dim3(kSrvBlock), lds, stream, a, cur,
                                   extend);
            };
            if (mode == kTravSingle) go(std::integral_constant<int, kTravSingle>{});
            else if (mode == kTravIdentity) go(std::integral_constant<int, kTravIdentity>{});
            else go(std::integral_constant<int, kTravGeneral>{});
        });
        if (extend) SOLHIP_HIP_CHECK(hipEventRecord(traced[cur], stream));
        timed(SOLHIP_KERNEL_SRV_SHADE, [&] {
            hipLaunchKernelGGL(k_srv_shade, dim3(shade_blocks), dim3(kSrvShadeBlock), 0, stream, a, cur, extend);
        });
        return srv_status("server step");
    }

    int step()
    {
        const int rc = launch((uint32_t)(steps & 1u), 1u);
        ++steps;
        return rc;
    }

    // what the last step left for the next one besides its queue: its shadow rays
    // are answered and the slots that ended in it finished, so that a job is done after
    // as many steps as its longest pixel has segments
    int settle()
    {
        const uint32_t next = (uint32_t)(steps & 1u), last = next ^ 1u;
        if (std::all_of(running_by_idx.begin(), running_by_idx.end(), [](uint64_t id) { return id == 0; })) return 0;
        int rc = launch(next, 0u);
        if (!rc) rc = launch_fill(stream, (uint32_t *)counts.ptr + (2 + last) * kCount, 1, 0u);
        if (!rc) rc = launch_fill(stream, (uint32_t *)counts.ptr + (4 + last) * kCount, 1, 0u);
        return rc;
    }

    // the jobs whose done counters, as of the start of step `at`, are full give back their slots
    void finish_jobs(const uint32_t *counts, uint64_t at)
    {
        const double t = now_ms(t0);
        for (uint32_t j = 0; j < max_jobs; ++j) {
            const uint64_t id = running_by_idx[j];
            if (!id) continue;
            SrvJob &jb = all[id];
            if (jb.first_step <= at && counts[j] >= jb.npix) {
                jb.state = SOLHIP_JOB_DONE;
                jb.t_done = t;
                free_range(jb.base, jb.slots);
                running_by_idx[j] = 0;
            }
        }
    }

    // the counters that step `at` wrote at its start
    int poll_step(uint64_t at)
    {
        SOLHIP_HIP_CHECK(hipEventSynchronize(traced[at & 1u]));
        finish_jobs(done_host + (at & 1u) * max_jobs, at);
        return 0;
    }

    // the counters now, once all launched steps are complete
    int poll()
    {
        uint32_t *now = done_host + 2 * max_jobs;
        SOLHIP_HIP_CHECK(hipMemcpyAsync(now, done.ptr, sizeof(uint32_t) * max_jobs, hipMemcpyDeviceToHost, stream));
        SOLHIP_HIP_CHECK(hipStreamSynchronize(stream));
        finish_jobs(now, steps);
        return 0;
    }
    uint32_t live() const
    {
        uint32_t n = (uint32_t)waiting.size();
        for (uint64_t id : running_by_idx) n += id ? 1u : 0u;
        return n;
    }
};

}  // namespace solhip

using namespace solhip;

extern "C" {

int32_t solhip_server_create(solhip_ctx ctx, uint64_t hbm_budget, uint32_t max_jobs, solhip_server *out)
{
    Context *c = ctx_of(ctx);
    if (!c) return bad_handle("context");
    if (!out) return bad_arg("out");
    if (max_jobs == 0 || max_jobs > kMaxJobs) return bad_arg("max_jobs must be in [1, 256]");
    const uint64_t slots = hbm_budget / kSlotBytes;
    if (slots < 64 || slots > 0xFFFFFF00ull) return bad_arg("HBM budget out of range");
    Server *sv = new Server();
    sv->kind = Kind::Server;
    sv->ctx = ctx;
    sv->cx = c;
    sv->max_slots = (uint32_t)slots;
    sv->max_jobs = max_jobs;
    sv->running_by_idx.assign(max_jobs, 0);
    sv->free_ranges[0] = sv->max_slots;
    sv->t0 = std::chrono::steady_clock::now();
    const uint64_t n = slots;
    bool fail = sv->jobs.reserve((uint64_t)max_jobs * sizeof(JobDev)) || sv->st0.reserve(n * 16) ||
                sv->st1.reserve(n * 16) || sv->psum.reserve(n * 16) || sv->fsum.reserve(n * sizeof(FixSum)) ||
                sv->pmeta.reserve(n * 4) ||
                sv->q0.reserve(n * sizeof(QRay)) || sv->q1.reserve(n * sizeof(QRay)) ||
                sv->hits.reserve(n * sizeof(QHit)) || sv->sq.reserve(n * sizeof(QRay)) ||
                sv->scontrib.reserve(n * 16) || sv->finished.reserve(n * 4) || sv->counts.reserve(6ull * kCount * 4) ||
                sv->heads.reserve((uint64_t)kFetchWords * 4) || sv->done.reserve((uint64_t)max_jobs * 4);
    if (!fail) fail = hipStreamCreateWithFlags(&sv->stream, hipStreamNonBlocking) != hipSuccess ||
                      hipHostMalloc((void **)&sv->done_host, 3 * sizeof(uint32_t) * max_jobs, hipHostMallocDefault) !=
                          hipSuccess ||
                      hipEventCreateWithFlags(&sv->traced[0], hipEventDisableTiming) != hipSuccess ||
                      hipEventCreateWithFlags(&sv->traced[1], hipEventDisableTiming) != hipSuccess;
    if (fail) {
        sv->release_all();
        delete sv;
        set_error("render server allocation failed");
        return SOLHIP_ERROR_OUT_OF_MEMORY;
    }
    if (launch_fill(sv->stream, (uint32_t *)sv->counts.ptr, 6ull * kCount, 0u) ||
        launch_fill(sv->stream, (uint32_t *)sv->heads.ptr, (uint64_t)kFetchWords, 0u) ||
        launch_fill(sv->stream, (uint32_t *)sv->done.ptr, max_jobs, 0u) || hipStreamSynchronize(sv->stream)) {
        sv->release_all();
        delete sv;
        return SOLHIP_ERROR_DEVICE;
    }
    *out = reg(sv);
    return SOLHIP_OK;
}

int32_t solhip_server_destroy(solhip_ctx ctx, solhip_server h)
{
    Context *c = ctx_of(ctx);
    if (!c) return bad_handle("context");
    Server *sv = static_cast<Server *>(unreg(h, Kind::Server));
    if (!sv) return bad_handle("server");
    (void)hipStreamSynchronize(sv->stream);
    sv->release_all();
    delete sv;
    return SOLHIP_OK;
}

// the scene's TLAS still exists with the generation it had at registration,
// and its BLASes are those it was built over
static int scene_fresh(const SrvScene *sc)
{
    const Tlas *t = get<Tlas>(sc->tlas, Kind::Tlas);
    if (!t || t->gen != sc->tlas_gen) {
        set_error(std::string("the scene's TLAS was ") + (t ? "rebuilt" : "destroyed") +
                  " after solhip_server_scene registered it; register the scene again");
        return SOLHIP_ERROR_STALE;
    }
    return check_fresh(t);
}

int32_t solhip_server_scene(solhip_ctx ctx, solhip_server h, solhip_tlas th, const solhip_scene_tables *tables,
                            uint32_t *scene_id)
{
    Context *c = ctx_of(ctx);
    if (!c) return bad_handle("context");
    Server *sv = get<Server>(h, Kind::Server);
    if (!sv) return bad_handle("server");
    Tlas *t = get<Tlas>(th, Kind::Tlas);
    if (!t) return bad_handle("TLAS");
    if (!tables || !tables->instances_addr || !tables->vertex_table_addr || !tables->index_table_addr ||
        !tables->material_table_addr || (tables->index_size != 4 && tables->index_size != 8) || !scene_id)
        return bad_arg("scene tables");
    if (const int rc = check_fresh(t)) return rc;
    if (stack_depth_of(t) > (uint32_t)kMaxStack) {
        set_error("acceleration structures too deep for the traversal stack");
        return SOLHIP_ERROR_UNSUPPORTED;
    }
    SrvScene *sc = new SrvScene();
    sc->sv = view_of(t);
    sc->tlas = th;
    sc->tlas_gen = t->gen;
    sc->identity = t->identity;
    sc->tb.instances = (const solhip_scene_instance *)tables->instances_addr;
    sc->tb.vertex_table = (const uint64_t *)tables->vertex_table_addr;
    sc->tb.index_table = (const uint64_t *)tables->index_table_addr;
    sc->tb.material_table = (const uint64_t *)tables->material_table_addr;
    sc->tb.instance_count = tables->instance_count;
    sc->tb.index_size = tables->index_size;
    uint32_t nl = 0;
    int rc = build_lights(sv->stream, sc->tb, t, sc->light_offsets, sc->lights, &nl, nullptr);
    if (rc) {
        sc->light_offsets.release();
        sc->lights.release();
        delete sc;
        return rc;
    }
    sc->nlights = nl;
    if (nl) {
        LightTri last;
        SOLHIP_HIP_CHECK(hipMemcpyAsync(&last, (const LightTri *)sc->lights.ptr + (nl - 1), sizeof(LightTri),
                                        hipMemcpyDeviceToHost, sv->stream));
        SOLHIP_HIP_CHECK(hipStreamSynchronize(sv->stream));
        sc->total = last.cdf;
    }
    sv->max_stack = std::max(sv->max_stack, sc->sv.stack_depth);
    sv->scenes.push_back(sc);
    *scene_id = (uint32_t)(sv->scenes.size() - 1);
    return SOLHIP_OK;
}

int32_t solhip_server_submit(solhip_ctx ctx, solhip_server h, const solhip_job_desc *job, uint64_t *job_id)
{
    Context *c = ctx_of(ctx);
    if (!c) return bad_handle("context");
    Server *sv = get<Server>(h, Kind::Server);
    if (!sv) return bad_handle("server");
    if (!job || !job_id) return bad_arg("job");
    if (job->scene >= sv->scenes.size()) return bad_arg("scene id");
    if (const int rc = scene_fresh(sv->scenes[job->scene])) return rc;
    if (job->W == 0 || job->H == 0) return bad_arg("image size");
    const uint64_t npix = (uint64_t)job->W * job->H;
    if (job->spec.sample_streams && (uint64_t)job->spec.spp_per_frame * npix > (1ull << 32))
        return bad_arg("sample_streams: spp_per_frame * W * H must not exceed 2^32");
    if (npix > sv->max_slots) return bad_arg("image larger than the server's slot budget");
    if (job->spec.spp_per_frame == 0 || job->spec.spp_per_frame > 0xFFFFFFu || job->spec.max_depth > 4096 ||
        job->spec.enable_sky > 2 || job->spec.sample_streams > 1)
        return bad_arg("job spec");
    Buffer *acc = get<Buffer>(job->accum, Kind::Buffer);
    if (!acc || acc->bytes < npix * 16) return bad_arg("job accum buffer");
    if (job->out_rgba8) {
        Buffer *o = get<Buffer>(job->out_rgba8, Kind::Buffer);
        if (!o || o->bytes < npix * 4) return bad_arg("job out_rgba8 buffer");
    }
    SrvJob jb;
    jb.desc = *job;
    jb.npix = (uint32_t)npix;
    if (job->spec.sample_streams) {
        const uint32_t spp = job->spec.spp_per_frame;
        uint64_t lanes = job->spec.wf_samples_per_pass;
        if (lanes == 0)
            lanes = std::min<uint64_t>((spp + kLaneSamples - 1) / kLaneSamples, std::max<uint64_t>(1, kJobSlots / npix));
        lanes = std::max<uint64_t>(1, std::min<uint64_t>({lanes, spp, sv->max_slots / npix}));
        jb.lanes_max = (uint32_t)lanes;
    }
    jb.t_submit = now_ms(sv->t0);
    const uint64_t id = sv->next_id++;
    sv->all[id] = jb;
    sv->waiting.push_back(id);
    *job_id = id;
    return SOLHIP_OK;
}

int32_t solhip_server_run(solhip_ctx ctx, solhip_server h, uint32_t max_steps, uint32_t *live)
{
    Context *c = ctx_of(ctx);
    if (!c) return bad_handle("context");
    Server *sv = get<Server>(h, Kind::Server);
    if (!sv) return bad_handle("server");
    // a scene rebuilt since its registration would leave jobs reading freed
    // or changed acceleration structures: refuse to run them
    for (const auto &kv : sv->all) {
        const SrvJob &jb = kv.second;
        if (jb.state == SOLHIP_JOB_DONE) continue;
        if (const int rc = scene_fresh(sv->scenes[jb.desc.scene])) return rc;
    }
    // The host stays a step ahead of the GPU: it looks at the done counters of the
    // step before the one that it has just launched.
    const uint64_t begin = sv->steps;
    bool running = false;
    int rc = 0;
    for (uint32_t k = 0; k < max_steps && !rc; ++k) {
        rc = sv->admit();
        if (rc) break;
        running = false;
        for (uint64_t id : sv->running_by_idx) running = running || id != 0;
        if (!running) break;
        rc = sv->step();
        if (!rc && sv->steps >= begin + 2) rc = sv->poll_step(sv->steps - 2);
    }
    // no step is in flight on return, with an error neither
    if (sv->steps != begin) {
        if (!rc && running) rc = sv->settle();
        const int polled = sv->poll();
        if (!rc) rc = polled;
    }
    if (rc) return rc;
    if (live) *live = sv->live();
    return SOLHIP_OK;
}

int32_t solhip_server_job(solhip_ctx ctx, solhip_server h, uint64_t job_id, solhip_job_status *out)
{
    Context *c = ctx_of(ctx);
    if (!c) return bad_handle("context");
    Server *sv = get<Server>(h, Kind::Server);
    if (!sv) return bad_handle("server");
    auto it = sv->all.find(job_id);
    if (it == sv->all.end() || !out) return bad_arg("job id");
    std::memset(out, 0, sizeof(*out));
    out->state = it->second.state;
    out->submit_ms = it->second.t_submit;
    out->admit_ms = it->second.t_admit;
    out->done_ms = it->second.t_done;
    return SOLHIP_OK;
}

}  // extern "C"
