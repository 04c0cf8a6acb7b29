// modes_cpu.hip -- the step traversal in a given form (kTravGeneral,
// kTravSingle, kTravIdentity) on the host, for the CPU test that compares the
// forms.  Test infrastructure: not part of libsolhip.
#include "bvh_cpu.hip"

namespace {

template <bool ANY, int MODE>
void run_mode(HostScene *s, const SceneView &sv, const float *r, uint2 *lds, TravCounts &tc, Hit &hit)
{
    TravState st;
    trav_init<MODE, true>(st, sv, v3(r[0], r[1], r[2]), v3(r[4], r[5], r[6]), r[3], r[7], 0xFFu, tc);
    while (!trav_step<ANY, true, true, MODE>(st, sv, 0xFFu, lds, 1, tc)) {
    }
    hit = trav_result(st);
}

}  // namespace

extern "C" void hc_trace_mode(void *h, const float *rays, uint32_t n, uint32_t any, uint32_t mode, void *hits,
                              uint64_t *counts)
{
    HostScene *s = static_cast<HostScene *>(h);
    SceneView sv{};
    sv.tnodes = s->insts.empty() ? nullptr : s->tlas.nodes.data();
    sv.insts = s->insts.data();
    sv.single = s->insts.size() == 1 ? 1u : 0u;
    sv.inst_meta = s->meta.data();
    uint32_t max_blas_depth = 0;
    for (const auto &b : s->blas) max_blas_depth = std::max(max_blas_depth, b.bvh.depth);
    sv.stack_depth = std::min<uint32_t>(kMaxStack, s->tlas.depth + max_blas_depth + 1) + 2;
    uint2 lds[kMaxStack + 2];
    for (uint32_t i = 0; i < n; ++i) {
        const float *r = rays + 8 * (size_t)i;
        TravCounts tc{0, 0, 0, false};
        Hit hit;
        if (mode == kTravSingle)
            any ? run_mode<true, kTravSingle>(s, sv, r, lds, tc, hit) : run_mode<false, kTravSingle>(s, sv, r, lds, tc, hit);
        else if (mode == kTravFew)
            any ? run_mode<true, kTravFew>(s, sv, r, lds, tc, hit) : run_mode<false, kTravFew>(s, sv, r, lds, tc, hit);
        else if (mode == kTravIdentity)
            any ? run_mode<true, kTravIdentity>(s, sv, r, lds, tc, hit) : run_mode<false, kTravIdentity>(s, sv, r, lds, tc, hit);
        else
            any ? run_mode<true, kTravGeneral>(s, sv, r, lds, tc, hit) : run_mode<false, kTravGeneral>(s, sv, r, lds, tc, hit);
        put_hit(hits, i, hit);
        counts[0] += tc.nodes;
        counts[1] += tc.tris;
        counts[2] += tc.insts;
        counts[3] += tc.overflow ? 1 : 0;
    }
}
