// Host-only checks of the tiled kernels' plan (nuvec_amd/csrc/nvq_splits.h), compiled and run by tests/test_host_tiles.py: the choices
// among timed tiles and splits of K for 256 compute units, and what the kernels take for granted, over a grid of shapes, formats and chip
// sizes: every plan has it, and a plan without it is named before a launch.
#include <stdio.h>
#include <string.h>

#include "nuvec_hip.h"
#include "nvq_splits.h"

using namespace nvq::splits;

static long g_failures = 0, g_plans = 0;
#define EXPECT(cond, ...)                                      \
    do {                                                       \
        if (!(cond)) {                                         \
            if (g_failures++ < 20) {                           \
                printf("FAILED %s: ", #cond);                  \
                printf(__VA_ARGS__);                           \
                printf("\n");                                  \
            }                                                  \
        }                                                      \
    } while (0)

// Products timed on every tile and split (microseconds on MI355X): the plan is one of the timed ones, at most a tenth above the
// fastest, and its estimate a quarter off at most.
struct Timed {
    int tile, want;  // `want`: the parts of K that were asked for (in whole windows there may be fewer)
    double us;
};
struct Case {
    int mode, bits;
    bool float16, exact;
    int64_t m, n, k;
    Timed timed[6];
};
static const Case cases[] = {
    // K beyond 14336, few tiles
    {NVQ_MXFP4, 4, false, false, 79, 4165, 21632, {{kQmk128, 7, 34.3}, {kQmk128, 6, 36.5}, {kQmk128, 5, 38.7}, {kQmk128, 4, 46.0}, {kQmk64, 3, 46.3}, {kQmk128, 8, 48.8}}},
    {NVQ_MXFP4, 4, false, false, 128, 3488, 18784, {{kQmk128, 8, 30.4}, {kQmk128, 7, 31.2}, {kQmk64, 4, 33.3}, {kQmk128, 6, 33.7}, {kQmk64, 8, 38.1}, {kQmk128, 4, 42.8}}},
    {NVQ_MXFP8, 8, false, false, 236, 1161, 22656, {{kQmk128, 8, 34.9}, {kQmk64, 5, 35.7}, {kQmk128, 7, 35.9}, {kQmk64, 6, 36.6}, {kQmk128, 6, 38.5}, {kQmk64, 4, 40.7}}},
    {NVQ_NVFP4, 4, false, false, 592, 701, 18944, {{kQmk128, 6, 38.3}, {kQmk128, 8, 39.6}, {kQmk64, 4, 40.5}, {kQmk128, 7, 41.1}, {kQmk64, 8, 46.9}, {kQmk128, 4, 47.7}}},
    {NVQ_NVFP4, 4, false, false, 512, 4096, 32288, {{kBig, 8, 149.3}, {kQmk128, 2, 154.9}, {kBig, 7, 158.1}, {kQmk128, 4, 159.3}, {kQmk128, 6, 172.4}, {kQmk128, 8, 177.8}}},
    {NVQ_AFFINE, 4, true, false, 354, 1072, 18944, {{kQmk128, 7, 37.6}, {kQmk128, 8, 37.8}, {kQmk128, 6, 37.9}, {kQmk64, 4, 41.9}, {kQmk128, 4, 47.5}, {kQmk64, 8, 49.3}}},
    {NVQ_AFFINE, 3, false, true, 128, 3848, 31552, {{kQmk128, 8, 54.3}, {kQmk128, 7, 58.1}, {kQmk128, 6, 64.1}, {kQmk64, 4, 83.2}, {kQmk128, 4, 87.3}, {kQmk64, 8, 88.9}}},
    {NVQ_AFFINE, 8, false, true, 143, 2438, 28672, {{kQmk128, 6, 57.8}, {kQmk128, 5, 63.7}, {kQmk64, 4, 63.9}, {kQmk64, 8, 70.1}, {kQmk128, 4, 73.8}, {kQmk128, 8, 81.1}}},
    // short K, one round of 128 x 128 tiles and several of the others
    {NVQ_AFFINE, 6, false, false, 256, 31806, 64, {{kSmall, 1, 8.8}, {kQmk128, 1, 16.5}, {kBig, 1, 17.0}, {kQmk64, 1, 20.3}}},
    {NVQ_AFFINE, 8, false, false, 256, 14813, 704, {{kSmall, 1, 14.0}, {kQmk128, 1, 14.8}, {kQmk64, 1, 19.1}, {kBig, 1, 28.6}}},
    {NVQ_MXFP4, 4, true, false, 69, 24262, 384, {{kSmall, 1, 8.8}, {kQmk128, 1, 9.8}, {kQmk64, 1, 11.6}, {kBig, 1, 21.5}}},
    {NVQ_MXFP8, 8, false, false, 79, 31563, 320, {{kSmall, 1, 9.1}, {kQmk128, 1, 10.0}, {kQmk64, 1, 12.1}, {kBig, 1, 21.7}}},
    {NVQ_AFFINE, 8, false, true, 1024, 3717, 576, {{kQmk128, 1, 13.8}, {kSmall, 1, 14.6}, {kQmk64, 1, 18.1}}},
    // few outputs
    {NVQ_AFFINE, 5, false, true, 412, 1024, 4096, {{kQmk128, 8, 21.2}, {kQmk64, 5, 22.2}, {kQmk64, 4, 22.2}, {kQmk128, 7, 23.0}, {kQmk128, 6, 23.1}, {kQmk64, 8, 27.1}}},
};

static int parts_of(int64_t steps, int want) {
    const int64_t per = ((steps + want - 1) / want + 3) & ~(int64_t)3;
    return want == 1 ? 1 : (int)((steps + per - 1) / per);
}

int main() {
    for (const Case &c : cases) {
        const Product a{c.m, c.n, c.k, 1, false, c.exact, step_times(c.mode, c.bits, c.float16, c.exact)};
        const Plan p = qmm_plan(a, 256);
        double best = 1e30, chosen = 1e30;
        for (const Timed &t : c.timed) {
            if (t.us == 0.0) continue;
            if (t.us < best) best = t.us;
            if (t.tile == p.tile && parts_of(p.units, t.want) == p.splits) chosen = t.us;
        }
        g_plans++;
        EXPECT(chosen <= 1.1 * best, "mode %d, %d bits, %lld rows, W[%lld,%lld]: tile %d in %d parts takes %.1f us, the fastest %.1f", c.mode, c.bits, (long long)c.m,
               (long long)c.n, (long long)c.k, p.tile, p.splits, chosen, best);
        // (the routes weigh it against the other kernels' times)
        EXPECT(p.estimate_us > 0.8 * best && p.estimate_us < 1.25 * best, "mode %d, %d bits, %lld rows, W[%lld,%lld]: estimated %.1f us, takes %.1f", c.mode, c.bits,
               (long long)c.m, (long long)c.n, (long long)c.k, p.estimate_us, best);
    }
    struct { int mode, bits; } formats[] = {{NVQ_AFFINE, 1}, {NVQ_AFFINE, 3}, {NVQ_AFFINE, 4}, {NVQ_AFFINE, 5}, {NVQ_MXFP4, 4}, {NVQ_MXFP8, 8}, {NVQ_NVFP4, 4}};
    const int64_t ms[] = {5, 17, 33, 64, 65, 129, 300, 640, 641, 2048, 5000000}, ns[] = {8, 129, 1000, 4096, 8192, 32768}, batches[] = {1, 3, 64};
    const int64_t ks[] = {64, 96, 128, 512, 544, 1056, 1088, 4096, 7200, 14336, 14400, 16384, 16416, 32768, 65536};
    for (auto f : formats) for (int float16 = 0; float16 < 2; float16++) for (int exact = 0; exact <= (f.mode == NVQ_AFFINE); exact++)
        for (int64_t m : ms) for (int64_t n : ns) for (int64_t k : ks) for (int64_t b : batches) for (int cus : {1, 64, 256, 304}) {
            if (k % kQmmStep != 0 && f.mode == NVQ_AFFINE && !exact) continue;  // (no product of the tiled kernels)
            const Product a{m, n, k, b, false, exact != 0, step_times(f.mode, f.bits, float16 != 0, exact != 0)};
            const Plan p = qmm_plan(a, cus);
            g_plans++;
            const char *fault = qmm_plan_fault(p, a);
            EXPECT(fault == nullptr, "%s: mode %d, m=%lld n=%lld k=%lld batch=%lld cus=%d", fault, f.mode, (long long)m, (long long)n, (long long)k, (long long)b, cus);
            EXPECT(p.splits <= 8 && (p.splits == 1 || b == 1), "%d parts", p.splits);
            EXPECT(!exact || p.tile != kBig, "256 x 256 with two roundings");
            EXPECT(p.tile != kQmk64 || (m + 63) / 64 <= 65535, "%lld rows in tiles of 64", (long long)m);
            if (k <= 14336 || k % kQmmStep != 0)
                EXPECT(workspace_bytes(p, a) <= (size_t)NVQ_STATIC_SCRATCH_BYTES, "m=%lld n=%lld k=%lld: %zu bytes of partial sums", (long long)m, (long long)n, (long long)k, workspace_bytes(p, a));
        }
    const Product plain{300, 700, 4096, 1, false, false}, exact{300, 700, 4096, 1, false, true}, batch{300, 700, 4096, 2, false, false}, half{300, 700, 4128, 1, false, true};
    const Product exact_batch{300, 700, 4096, 2, false, true};
    EXPECT(qmm_plan_fault(Plan{1, 64, 64, 0.0, kQmk128}, plain) == nullptr && qmm_plan_fault(Plan{2, 32, 64, 0.0, kQmk64}, plain) == nullptr, "sound plans");
    EXPECT(qmm_plan_fault(Plan{1, 64, 64, 0.0, kSmall}, exact) == nullptr, "a sound plan");
    EXPECT(qmm_plan_fault(Plan{5, 16, 64, 0.0, kQmk128}, plain) != nullptr, "a fifth part of four");
    EXPECT(qmm_plan_fault(Plan{3, 23, 64, 0.0, kQmk128}, plain) != nullptr, "parts of half a window");
    EXPECT(qmm_plan_fault(Plan{1, 63, 63, 0.0, kQmk128}, plain) != nullptr, "steps of another K");
    EXPECT(qmm_plan_fault(Plan{2, 32, 64, 0.0, kQmk128}, batch) != nullptr, "a split batch");
    EXPECT(qmm_plan_fault(Plan{1, 64, 64, 0.0, kBig}, exact) != nullptr, "256 x 256 with two roundings");
    EXPECT(qmm_plan_fault(Plan{1, 65, 65, 0.0, kSmall}, half) != nullptr && qmm_plan_fault(Plan{1, 64, 64, 0.0, kSmall}, exact_batch) != nullptr, "steps and a half, a batch");
    printf("%ld plans checked, %ld failures\n", g_plans, g_failures);
    return g_failures != 0;
}
