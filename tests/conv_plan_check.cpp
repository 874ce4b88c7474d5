// Host harness of conv_plan (mf-lbm-cuda_amd/csrc/conv_plan.h) for tests/test_conv_plan.py.  Built
// with g++ (the header's device qualifiers defined away).  Arguments D H W cin cout: prints the
// chosen box and its launch, and checks the coordinates that the kernel takes from a block's index
// against division.  Exit status: 0, 1 no box, 2 wrong coordinates, 3 boxes that miss voxels or do
// not fit, 4 arguments.  With the one argument "kept": plans kept by size against searches, for sizes
// that come back and sizes that take each other's places (exit status 5 where they differ, 6 where a
// size that just came is searched for again).
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include "conv_plan.h"

static int kept() {
    uint32_t x = 7;
    auto draw = [&](int lo, int hi) { return lo + (int)((x = x * 1664525u + 1013904223u) >> 8) % (hi - lo + 1); };
    for (int i = 0; i < 20000; ++i) {
        const mfnn::Grid3 g{draw(1, 12), draw(1, 12), draw(1, 12)};
        const int cin = 8 * draw(1, i % 50 ? 6 : 150), ntw = draw(1, 4);
        mfnn::ConvPlan want;
        const bool found = mfnn::conv_plan(g, cin, ntw, want);
        const mfnn::ConvPlan* got = mfnn::kept_plan(g, cin, ntw);
        if (found != (got != nullptr)) return 5;
        if (!got) continue;
        if (got->t.tx != want.t.tx || got->t.ty != want.t.ty || got->t.tz != want.t.tz || got->t.pu != want.t.pu ||
            got->t.dnx.mul != want.t.dnx.mul || got->t.dny.shift != want.t.dny.shift || got->mt != want.mt ||
            got->nt != want.nt || got->lds != want.lds || got->boxes != want.boxes)
            return 5;
        // a mark in the kept plan is still there
        const_cast<mfnn::ConvPlan*>(got)->t.tv += 1000;
        if (mfnn::kept_plan(g, cin, ntw)->t.tv != want.t.tv + 1000) return 6;
        const_cast<mfnn::ConvPlan*>(got)->t.tv -= 1000;
    }
    return 0;
}

int main(int argc, char** argv) {
    if (argc == 2 && !std::strcmp(argv[1], "kept")) return kept();
    if (argc != 6) return 4;
    const mfnn::Grid3 g{std::atoi(argv[1]), std::atoi(argv[2]), std::atoi(argv[3])};
    const int cin = std::atoi(argv[4]), ntw = (std::atoi(argv[5]) + 15) / 16;
    mfnn::ConvPlan p;
    if (!mfnn::conv_plan(g, cin, ntw, p)) return 1;
    const mfnn::ConvTile& t = p.t;
    std::printf("%d %d %d mt %d nt %d lds %zu boxes %u\n", t.tx, t.ty, t.tz, p.mt, p.nt, p.lds, p.boxes);
    const int64_t nz = (g.D + t.tz - 1) / t.tz;
    if ((int64_t)p.boxes != (int64_t)t.nx * t.ny * nz || (int64_t)t.nx * t.tx < g.W || (int64_t)t.ny * t.ty < g.H) return 3;
    if (p.lds > 160 * 1024 || 64 * p.mt < t.tv || t.tv != t.tx * t.ty * t.tz || p.nt > ntw) return 3;
    // every block of small launches; of large ones, runs at both ends and a stride prime to the sides
    const int64_t n = p.boxes, step = n < 3000000 ? 1 : 101;
    for (int64_t b = 0; b < n; b += (b < 100000 || b > n - 100000) ? 1 : step) {
        const int yz = quot((int)b, t.dnx), bz = quot(yz, t.dny);
        if (yz != b / t.nx || bz != yz / t.ny) return 2;
    }
    return 0;
}
