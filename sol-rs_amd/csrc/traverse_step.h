// traverse_step.h -- the two-level traversal of traverse.h as a resumable
// state machine: trav_step does one step of work (at most one triangle, one
// instance entry and one node, with the stack pops between them) and reports
// when the ray is done.
// A lane whose ray has finished can then take the next ray while the rest of
// its wave keeps traversing (persistent threads with per-lane refill), which
// is what incoherent rays (AO, bounces) need to keep the SIMD busy.
//
// The visit order is exactly trace_ray's: instance leaves before descending,
// a BLAS traversed to the end before the TLAS continues (the TLAS state is
// pushed as two stack entries, the pending node group and then the pending
// instance-leaf group, tagged in bit 31), so closest and first hits equal
// trace_ray's bit for bit.
//
// Four forms of it, by what the TLAS holds (SceneView::mode, decided when the
// TLAS is built):
//   kTravGeneral   any scene.
//   kTravSingle    one instance: the ray enters it when it starts, in object space
//                  from then on, so a step has no TLAS phase, no instance entry and
//                  no way back, and the state no world ray.
//   kTravIdentity  every instance at the identity transform (a scene whose
//                  transforms are baked into its vertices): the object ray is the same
//                  in every instance, so it and its divisions are made once per
//                  ray and an instance entry only switches node arrays.
//   kTravFew       kTravIdentity in trees of at most kFewLevels levels (a room of a few
//                  boxes), whose nodes lead to many triangles each: trav_step's MORE.
// An instance entry is 6 divisions and a 3x4 transform for the few lanes of a
// wave that are at one, in almost every step, and the world ray 9 registers
// (k_trace_rays 89 -> 70 VGPRs).  One instance of 2.1M triangles: AO frame 3.25
// -> 2.76 ms; 1.5M scattered rays 404 -> 354 us; the Cornell box's six: 16-spp
// path-traced frame 5.5 -> 5.2 ms.
// All give the same hits and fetch counts.
#pragma once

#include "traverse.h"

namespace solhip {

struct TravState {
    V3 wo, wd, winv;           // world ray and its safe_inv direction
    V3 o, inv;                 // ray of the current level (object space inside a BLAS)
    Wt wt;                     // triangle test of the current BLAS ray
    float tmin, tlo;
    uint32_t oct;
    uint32_t level;            // 0: TLAS, 1: BLAS
    uint32_t inst;             // instance index of the BLAS being traversed
    const WideNode *nodes;     // BLAS nodes
    const TriRec *tris;        // BLAS leaf records
    uint32_t ng_base, ng_hits, ng_imask;
    uint32_t tg_base, tg_mask, tg_valid;   // leaf group: first record, primitives left, the node's leaf_mask
    int sp, base;              // stack height; height at BLAS entry
    Hit best;
    bool any;                  // first hit ends the ray (with kAnyOfRay only)
};

// trav_step's ANY: closest hit, first hit, or as the ray says (TravState::any)
constexpr int kClosest = 0, kAny = 1, kAnyOfRay = 2;

constexpr int kMoreByScene = -1;   // trav_step's MORE

// the form whose phases a form has
constexpr int form_of(int form) { return form == kTravFew ? kTravIdentity : form; }

constexpr uint32_t kLeafGroupTag = 0x80000000u;

// at least one in `of` of the wave's active lanes says yes, and one at all (the host has one lane)
SOLHIP_HD bool lanes_vote(bool yes, int of)
{
#ifdef __HIP_DEVICE_COMPILE__
    const uint64_t y = __ballot(yes);
    return y != 0 && __popcll(y) * of >= __popcll(__ballot(true));
#else
    (void)of;
    return yes;
#endif
}

// transforms the world ray into an instance and readies its triangle test
SOLHIP_HD void trav_object_ray(TravState &s, const float *m, V3 wo, V3 wd)
{
    const ObjectRay r = object_ray(m, wo, wd);
    s.o = r.o;
    s.inv = r.inv;
    s.oct = r.oct;
    s.wt = r.wt;
}

template <int FORM, bool COUNT>
SOLHIP_HD void trav_init(TravState &s, const SceneView &sv, V3 wo, V3 wd, float tmin, float tmax, uint32_t cull,
                         TravCounts &cnt)
{
    constexpr int MODE = form_of(FORM);
    s.wo = wo;
    s.wd = wd;
    s.tmin = tmin;
    s.tlo = tmin - fabsf(tmin) * 0x1p-20f;
    s.level = 0;
    s.inst = 0;
    s.nodes = nullptr;
    s.tris = nullptr;
    s.tg_base = 0;
    s.tg_mask = 0;
    s.tg_valid = 1u;
    s.ng_base = 0;
    s.ng_hits = 0;
    s.ng_imask = 1u;
    s.sp = 0;
    s.base = 0;
    s.best.t = tmax;
    s.best.u = 0.0f;
    s.best.v = 0.0f;
    s.best.inst = SOLHIP_MISS;
    s.best.prim = SOLHIP_MISS;
    if (MODE == kTravSingle) {
        const uint32_t meta = SOLHIP_G1(sv.inst_meta)[0];
        const uint4 *ip = reinterpret_cast<const uint4 *>(sv.insts);
        const uint4 i0 = SOLHIP_G4(ip)[0], i1 = SOLHIP_G4(ip)[1], i2 = SOLHIP_G4(ip)[2], i3 = SOLHIP_G4(ip)[3];
        const uint64_t bn = ((uint64_t)i3.y << 32) | i3.x;
        const bool in = ((meta >> 24) & cull) != 0u;
        if (COUNT && in) cnt.insts++;
        const float m[12] = {as_f(i0.x), as_f(i0.y), as_f(i0.z), as_f(i0.w), as_f(i1.x), as_f(i1.y),
                             as_f(i1.z), as_f(i1.w), as_f(i2.x), as_f(i2.y), as_f(i2.z), as_f(i2.w)};
        trav_object_ray(s, m, wo, wd);
        s.nodes = reinterpret_cast<const WideNode *>(bn);
        s.tris = reinterpret_cast<const TriRec *>(((uint64_t)i3.w << 32) | i3.z);
        s.inst = meta & 0xFFFFFFu;
        s.level = 1;
        s.ng_hits = in && bn != 0 ? 1u << s.oct : 0u;   // nothing to enter: the first step ends the ray
    } else {
        if (MODE == kTravIdentity) {
            // the object ray has the bits of a transformed one; a zero's sign is
            // all that can differ from the world ray, and no box test depends on
            // that: the TLAS is traversed with the object ray, too
            trav_object_ray(s, kIdentityInverse, wo, wd);
        } else {
            s.o = wo;
            s.winv = safe_inv(wd);
            s.inv = s.winv;
            s.oct = octant(wd);
        }
        // the TLAS root, or, with one instance, its leaf (record 0) at once
        s.ng_hits = sv.tnodes && !sv.single ? (1u << s.oct) : 0u;
        s.tg_mask = sv.tnodes && sv.single ? 1u : 0u;
    }
}

SOLHIP_HD void trav_init(TravState &s, const SceneView &sv, V3 wo, V3 wd, float tmin, float tmax)
{
    TravCounts none{0, 0, 0, false};
    trav_init<kTravGeneral, false>(s, sv, wo, wd, tmin, tmax, 0xFFu, none);
}

// the final hit record of a finished traversal (trace_ray's miss convention)
SOLHIP_HD Hit trav_result(const TravState &s)
{
    Hit h = s.best;
    if (h.inst == SOLHIP_MISS) {
        h.t = -1.0f;
        h.u = 0.0f;
        h.v = 0.0f;
        h.prim = SOLHIP_MISS;
    }
    return h;
}

// One traversal step; true when the ray is finished.  A step does, in this
// order and each at most once: one triangle of the current leaf group, the
// BLAS exit and stack pop that lead to the next piece of work, one instance
// entry, one node test.  Running them as phases of one step (rather than one
// of them per step) lets a wave's lanes share the expensive node test in the
// same pass whatever bookkeeping each needed first.  lds: this lane's stack
// column, stride = lanes sharing the array, sv.stack_depth entries.
//
// WINV: a BLAS exit restores the world ray's inverse direction from the
// state (three more registers) instead of recomputing it (three correctly
// rounded divisions).  Measured per kernel: the AO kernels run 6 % faster
// with it; the path tracer's extension kernel, whose rays leave a BLAS 3.9
// times on average, 6 % faster once its register budget holds the three
// registers (at 5 waves per SIMD they spilled and it ran 1 % slower).
//
// A phase costs the wave its instructions however few lanes need it, so lanes vote:
// - An instance entry (general form: the transform, its six divisions) is taken by a few
//   lanes in almost every step: it waits until a quarter of the active lanes want
//   one (10,000 instances, a 1080p frame without its rebuild 53.4 -> 48.1 ms; 2M rays on 500
//   instances 1073 -> 973 us;
//   a half or a third or a sixth are 1 to 6 % slower; 8 lanes, not a share, hold up the last rays
//   of a launch: 0.2M rays 355 -> 415 us).
// - Lanes with triangles left sit out the node test, so the triangle phase is repeated
//   while one in MORE active lanes has another triangle (0: never).  kMoreByScene: 6 in trees
//   of a few levels (Cornell box: 2M rays 132 -> 104 us, 1080p AO 640 -> 555, path-traced
//   frame 3.38 -> 3.1 ms; 3 to 16 within 4 %), 3 in the general form (500 instances: 0.2M rays
//   353 -> 298 us, 2M 970 -> 911; 10,000: level), else never (terrain: 1 to 4 % slower, in one
//   instance or in 16 of 32K triangles).
// Which lane works when changes nothing for its ray: same visits, hits and counts.
template <int ANY, bool COUNT, bool WINV = true, int FORM = kTravGeneral, int MORE = kMoreByScene>
SOLHIP_HD bool trav_step(TravState &s, const SceneView &sv, uint32_t cull, uint2 *lds, int stride, TravCounts &cnt)
{
    constexpr int MODE = form_of(FORM);
    constexpr int more = MORE != kMoreByScene ? MORE : FORM == kTravFew ? 6 : FORM == kTravGeneral ? 3 : 0;
    const int depth = (int)sv.stack_depth;
    // 1. one triangle
    bool found = false;
    while (true) {
        const bool tri = (MODE == kTravSingle || s.level) && s.tg_mask && !found;
        if (tri) {
            const uint32_t k = __builtin_ctz(s.tg_mask);
            s.tg_mask &= s.tg_mask - 1u;
            const uint4 *tp = reinterpret_cast<const uint4 *>(s.tris + leaf_record(s.tg_base, s.tg_valid, k));
            const uint4 a = SOLHIP_G4(tp)[0], b = SOLHIP_G4(tp)[1];
            const uint2 c = SOLHIP_G2(tp + 2)[0];
            const float vv[9] = {as_f(a.x), as_f(a.y), as_f(a.z), as_f(a.w), as_f(b.x),
                                 as_f(b.y), as_f(b.z), as_f(b.w), as_f(c.x)};
            if (COUNT) cnt.tris++;
            float t, u, v;
            if (wt_hit(s.wt, s.tmin, s.best.t, vv, t, u, v) && better(t, s.inst, c.y, s.best)) {
                s.best.t = t;
                s.best.u = u;
                s.best.v = v;
                s.best.inst = s.inst;
                s.best.prim = c.y;
                found = ANY == kAny || (ANY == kAnyOfRay && s.any);
            }
        }
        // the lanes' vote: uniform, so they leave the loop together
        if (more == 0 || !lanes_vote(tri && s.tg_mask && !found, more)) break;
    }
    if (ANY != kClosest && found) return true;
    // 2. nothing left of the last node: the next stack entry (pushed groups are
    // never empty, so one pop leads to work).  An empty stack ends the ray at
    // once, also inside a BLAS: nothing of the TLAS is pending (its work is
    // pushed below the BLAS entry), so the world ray need not be restored.
    if (!s.tg_mask && !s.ng_hits) {
        if (s.sp == 0) return true;
        if (MODE != kTravSingle && s.level && s.sp == s.base) {
            // the BLAS is done: back to the world ray and the TLAS stack
            s.level = 0;
            if (MODE == kTravGeneral) {
                s.o = s.wo;
                s.inv = WINV ? s.winv : safe_inv(s.wd);
                s.oct = octant(s.wd);
            }
        }
        --s.sp;
        const uint2 e = lds[s.sp * stride];
        if (MODE != kTravSingle && (e.y & kLeafGroupTag)) {
            s.tg_base = e.x;
            s.tg_mask = e.y & ~kLeafGroupTag;
            s.tg_valid = 0xFFFFFFu;
        } else {
            s.ng_base = e.x;
            s.ng_hits = e.y & 0xFFu;
            s.ng_imask = (e.y >> 8) & 0xFFu;
        }
    }
    // 3. an instance leaf: enter its BLAS
    const bool enter = MODE != kTravSingle && !s.level && s.tg_mask;
    if ((MODE != kTravGeneral || lanes_vote(enter, 4)) && enter) {
        const uint32_t k = __builtin_ctz(s.tg_mask);
        s.tg_mask &= s.tg_mask - 1u;
        const uint32_t li = leaf_record(s.tg_base, s.tg_valid, k);
        const uint32_t meta = SOLHIP_G1(sv.inst_meta + li)[0];
        if (((meta >> 24) & cull) != 0u) {
            const uint4 *ip = reinterpret_cast<const uint4 *>(sv.insts + li);
            uint4 i0, i1, i2;
            if (MODE == kTravGeneral) {
                i0 = SOLHIP_G4(ip)[0];
                i1 = SOLHIP_G4(ip)[1];
                i2 = SOLHIP_G4(ip)[2];
            }
            const uint4 i3 = SOLHIP_G4(ip)[3];
            if (COUNT) cnt.insts++;
            const uint64_t bn = ((uint64_t)i3.y << 32) | i3.x;
            if (bn != 0) {
                // the TLAS continues later: pending node group, then pending leaves
                if (s.ng_hits) {
                    if (s.sp < depth) {
                        lds[s.sp * stride] = make_uint2(s.ng_base, s.ng_hits | (s.ng_imask << 8));
                        ++s.sp;
                    } else {
                        cnt.overflow = true;
                    }
                }
                if (s.tg_mask) {
                    // as record bits relative to the group's base
                    uint32_t left = 0;
                    for (uint32_t m = s.tg_mask; m; m &= m - 1u)
                        left |= 1u << leaf_record(0u, s.tg_valid, (uint32_t)__builtin_ctz(m));
                    if (s.sp < depth) {
                        lds[s.sp * stride] = make_uint2(s.tg_base, left | kLeafGroupTag);
                        ++s.sp;
                    } else {
                        cnt.overflow = true;
                    }
                }
                if (MODE == kTravGeneral) {
                    const float m[12] = {as_f(i0.x), as_f(i0.y), as_f(i0.z), as_f(i0.w), as_f(i1.x), as_f(i1.y),
                                         as_f(i1.z), as_f(i1.w), as_f(i2.x), as_f(i2.y), as_f(i2.z), as_f(i2.w)};
                    trav_object_ray(s, m, s.wo, s.wd);
                }
                s.nodes = reinterpret_cast<const WideNode *>(bn);
                s.tris = reinterpret_cast<const TriRec *>(((uint64_t)i3.w << 32) | i3.z);
                s.inst = meta & 0xFFFFFFu;
                s.level = 1;
                s.base = s.sp;
                s.ng_base = 0;
                s.ng_hits = 1u << s.oct;
                s.ng_imask = 1u;
                s.tg_base = 0;
                s.tg_mask = 0;
            }
        }
    }
    // 4. one node
    if (!s.tg_mask && s.ng_hits) {
        const uint32_t i = __builtin_ctz(s.ng_hits);
        s.ng_hits &= s.ng_hits - 1u;
        const uint32_t slot = i ^ s.oct;
        const uint32_t child = s.ng_base + __builtin_popcount(s.ng_imask & ((1u << slot) - 1u));
        if (s.ng_hits) {
            if (s.sp < depth) {
                lds[s.sp * stride] = make_uint2(s.ng_base, s.ng_hits | (s.ng_imask << 8));
                ++s.sp;
            } else {
                cnt.overflow = true;
            }
        }
        const WideNode *nodes = MODE == kTravSingle || s.level ? s.nodes : sv.tnodes;
        const uint4 *np = reinterpret_cast<const uint4 *>(nodes + child);
        const uint4 w0 = SOLHIP_G4(np)[0], w1 = SOLHIP_G4(np)[1], w2 = SOLHIP_G4(np)[2], w3 = SOLHIP_G4(np)[3],
                    w4 = SOLHIP_G4(np)[4];
        if (COUNT) cnt.nodes++;
        const float thi = s.best.t + fabsf(s.best.t) * 0x1p-20f;
        intersect_node(w0, w1, w2, w3, w4, s.o, s.inv, s.oct, s.tlo, thi, s.ng_hits, s.tg_mask);
        s.ng_base = w1.x;
        s.ng_imask = w0.w >> 24;
        s.tg_base = w1.y;
        s.tg_valid = w1.z;
    }
    return false;
}

}  // namespace solhip
