// The address and index widths a batched launch takes, per form (plan_views),
// on the host: octrees count as resident on device 0, which a hipGetDevice of
// this program's own reports.
#include <cstdio>

#include "view_desc.hpp"

extern "C" hipError_t hipGetDevice(int *device) {
    *device = 0;
    return hipSuccess;
}

int main() {
    using namespace svo;
    int bad = 0;
    auto expect = [&](bool ok, const char *what) {
        if (!ok) std::printf("wrong: %s\n", what);
        bad += !ok;
    };
    uint32_t resident = 0;
    svo_octree tight, loose;
    for (svo_octree *t : {&tight, &loose}) {
        t->words.assign(8, 0);
        t->depth = 11;
        t->levels = 10;
        t->device = 0;
        t->dwords = &resident;
    }
    loose.tight = false;
    svo_view v[2] = {};
    for (svo_view &w : v) {
        w.tree = &tight;
        w.width = w.height = 64;
        w.camera.tform[0] = w.camera.tform[5] = w.camera.tform[10] = 1.0f;
    }
    for (int both = 0; both < 2; ++both) {
        v[1].tree = both ? &loose : &tight;
        for (int form : {SVO_BATCH_GRID, SVO_BATCH_PERSISTENT}) {
            svo_batch_opts o{};
            o.form = form;
            ViewDesc hv[2];
            uint64_t htb[3];
            LaunchPlan plan;
            if (plan_views(v, 2, &o, 256, hv, htb, plan, false)) return 2;
            expect(plan.wide == (both && form == SVO_BATCH_GRID),
                   form == SVO_BATCH_GRID ? "grid form: 64-bit walk for a loose tree alone"
                                          : "persistent form: 32-bit indices for a loose tree too");
            if (form == SVO_BATCH_PERSISTENT)
                expect(plan.ldsPerBlock == size_t(plan.slots) * 64 * 8 * 4, "persistent form: 8 bytes per stack entry");
        }
    }
    const uint64_t k30 = uint64_t(1) << 30, k32 = uint64_t(1) << 32;
    expect(!wide_indices(k30) && !wide_indices(k32 - 1) && wide_indices(k32), "word indices: 32 bits below 2^32 words");
    std::printf("%s\n", bad ? "bad" : "ok");
    return bad;
}
