// Host harness of conv_plan (mf-lbm-cuda_amd/csrc/conv_plan.h) for tests/test_conv_plan.py.  Built
// with g++ (the header's device qualifiers defined away).  Arguments D H W cin cout: prints the
// chosen box and its launch, and checks the coordinates that the kernel takes from a block's index
// against division.  Exit status: 0, 1 no box, 2 wrong coordinates, 3 boxes that miss voxels or do
// not fit, 4 arguments.
#include <cstdio>
#include <cstdlib>
#include "conv_plan.h"

int main(int argc, char** argv) {
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
