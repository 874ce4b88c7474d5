// Boxes of the network's convolutions: the host's choice for a launch of k_conv3_box, with the
// quotients its kernels need, apart from the kernels so that the choice can be checked on a CPU.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <initializer_list>

namespace mfnn {

struct Grid3 {
    int D, H, W;
};

// Offset past what a buffer descriptor addresses (less than 2^31 bytes).
constexpr uint32_t NOWHERE = 0x80000000u;

// Exact quotients by a divisor fixed over a launch, without a branch: n / d =
// umulhi(n, ceil(2^32 / d)) while n * d < 2^32 (the launchers check it; in a box LDS bounds both);
// d = 1 passes n through the mask.
struct FastDiv {
    uint32_t d, mul, one;
};
inline FastDiv fast_div(uint32_t d) {
    return {d, d > 1 ? (uint32_t)(((1ull << 32) + d - 1) / d) : 0u, d > 1 ? 0u : ~0u};
}

// Exact quotients of any index below 2^31: n / d = n * ceil(2^(31 + l) / d) / 2^(31 + l) with
// 2^l >= d, in 64 bits.  For the index of a block, whose uniform product costs nothing: by FastDiv,
// grids of 65536 boxes and more had to be left to the gathering kernel (us, with it and on boxes:
// 256^3 48 -> 16 channels 5430 and 1400, 16 -> 48 6630 and 1045; 192^3 128 -> 128 81600 and 12800;
// 320^3 32 -> 32 14000 and 2470; smaller grids are level).
struct BlockDiv {
    uint32_t mul;
    int shift;
};
inline BlockDiv block_div(uint32_t d) {
    int l = 0;
    while ((1ull << l) < d) ++l;
    return {(uint32_t)(((1ull << (31 + l)) + d - 1) / d), 31 + l};
}
__host__ __device__ __forceinline__ int quot(int n, const BlockDiv& f) { return (int)((uint64_t)(uint32_t)n * f.mul >> f.shift); }

// What a workgroup of k_conv3_box needs of its box.
struct ConvTile {
    int tx, ty, tz, nx, ny;  // box, boxes along x and y
    int tv, pv;              // voxels of a box; of a loaded box, in whole groups of 16
    int pu;                  // 16-byte units of one loaded plane
    FastDiv row, c8, dtx, dty;  // units of a loaded row, of a voxel; tx, ty
    BlockDiv dnx, dny;          // nx, ny
};

// Channel tiles a wave may hold beside mt voxel tiles (registers).
inline int conv_max_nt(int mt) { return mt >= 8 ? 2 : mt >= 4 ? 3 : 4; }

// Box and tile counts of one k_conv3_box launch.
constexpr int64_t MAX_BOXES = (1 << 24) - 1;  // a launch holds fewer than 2^32 threads along x
struct ConvPlan {
    ConvTile t;
    int mt, nt;
    size_t lds;
    unsigned boxes;
};

// The gathering kernel (k_conv3) takes one channel tile per block where there are fewer blocks of
// four voxel tiles than CUs, or five and less per CU with one channel tile each; else all of them (us,
// one and all: 23040 voxels 1056 -> 32 503 and 587, 20480 720 -> 64 490 and 568, 25600 800 -> 64 785
// and 510, 32768 800 -> 64 976 and 515).
inline bool gather_single(const Grid3& g, int ntw) {
    const int64_t blocks = ((int64_t)g.D * g.H * g.W + 63) / 64;
    return blocks < 256 || (ntw > 1 && blocks * ntw <= 1280);
}

// Its time on more than 512 channels, in cycles: LDS then holds one workgroup of few voxels, whose
// box may cost more than it saves (us, gathered and on boxes: 32^3 800 -> 64 515 and 1430, 12^3 1056
// -> 128 395 and 604, 24^3 720 -> 64 381 and 440, 64^3 600 -> 128 5930 and 7360; 32^3 576 -> 64 529 and
// 480, 20^3 560 -> 128 338 and 227, 8^3 1056 -> 128 391 and 180).  A k block costs the latency of
// its loads or what the tiles move.
inline double gather_cycles(const Grid3& g, int cin, int ntw) {
    const double blocks = (double)(((int64_t)g.D * g.H * g.W + 63) / 64), nkb = (27 * (cin / 8) + 3) / 4;
    const double tiles = 1.3 * std::min(ntw, 4) + 0.7 * std::max(ntw - 4, 0);
    return nkb * (gather_single(g, ntw) ? 700.0 + blocks * ntw : std::max(2200.0, tiles * blocks));
}

// Box of a convolution: the equal splits of the axes with rows of up to 32 voxels are priced in
// cycles of a CU -- one per loaded 16-byte unit, the weights' 64 per channel tile and k block
// among them; per k block its MFMAs (16 each, a wave on each SIMD) and its operand reads (4 per
// wave and operand), at least the 70 of one block's dependent chain for a workgroup alone on
// its CU; load and MFMAs of two workgroups overlap where LDS holds both; whole rounds over the
// 256 CUs.  False where no box fits LDS or its launch, no descriptor a plane, or the gathering
// kernel is cheaper.
inline bool conv_plan(const Grid3& g, int cin, int ntw, ConvPlan& best) {
    const int c8 = cin / 8;
    const int nkb = (27 * c8 + 3) / 4;
    const size_t tab = (size_t)((nkb + 3) / 4 * 16 + 16) * 4;
    constexpr size_t LDS_MAX = 160 * 1024;
    double best_cost = 0.0;
    bool found = false;
    if (2ull * g.H * g.W * cin >= NOWHERE) return false;  // a plane that no descriptor addresses
    auto parts = [](int n, int lo, int hi, int* out) {  // the values ceil(n / p) in [lo, hi], largest first
        int cnt = 0;
        for (int v = std::min(n, hi); v >= 1 && (v >= lo || !cnt); --v) {
            const int p = (n + v - 1) / v;
            if ((n + p - 1) / p == v) out[cnt++] = v;
        }
        return cnt;
    };
    int xs[32], ys[8], zs[8];
    const int nxs = parts(g.W, 4, 32, xs), nys = parts(g.H, 1, 8, ys), nzs = parts(g.D, 1, 8, zs);
    // The largest splits, and beyond 256 channels, of which LDS holds small boxes only, all of them
    // (us, gathered, on boxes of the largest splits and of all: 128^3 320 -> 64 18800, none and 6170,
    // 64^3 448 -> 64 3290, none and 1750, 384 -> 128 5040, 5700 and 2400).
    const bool all = cin > 256;
    for (int a = 0; a < (all ? nxs : std::min(nxs, 6)); ++a)
        for (int b = 0; b < nys; ++b)
            for (int c = 0; c < (all ? nzs : std::min(nzs, 6)); ++c) {
                const int tx = xs[a], ty = ys[b], tz = zs[c], tv = tx * ty * tz;
                if (tv > 512) continue;
                const int mt = tv > 256 ? 8 : tv > 128 ? 4 : tv > 64 ? 2 : 1;
                const int64_t loaded = (int64_t)(tx + 2) * (ty + 2) * (tz + 2);
                const size_t lds_box = 16 * (1 + (size_t)((c8 + 1) / 2) * (2 * ((loaded + 15) / 16 * 16) + 1)) + tab;
                const int64_t boxes = (int64_t)((g.W + tx - 1) / tx) * ((g.H + ty - 1) / ty) * ((g.D + tz - 1) / tz);
                if (boxes > MAX_BOXES) continue;
                for (int nt = 1; nt <= 4 && nt <= ntw; ++nt) {
                    if (nt > conv_max_nt(mt)) continue;
                    const size_t lds = lds_box + 8192 * nt;
                    if (lds > LDS_MAX) continue;
                    const int64_t wgs = boxes * ((ntw + nt - 1) / nt);
                    const double load = (double)loaded * c8, fixed = 2000.0 + 250.0 * mt * nt;
                    const double block = std::max(std::max(16.0 * mt * nt, 16.0 * (mt + nt)), 64.0 * nt) + 24.0;
                    const double alone = load + nkb * std::max(block, 70.0) + fixed;
                    const double rounds = (double)((wgs + 255) / 256);
                    const double each = 2 * lds > LDS_MAX ? alone
                                                          : std::max(load, nkb * block) +
                                                                0.5 * std::min(load, nkb * block) + 0.5 * fixed;
                    const double cost = std::max(alone, rounds * each);
                    if (!found || cost < best_cost) {
                        found = true;
                        best_cost = cost;
                        best.t.tx = tx; best.t.ty = ty; best.t.tz = tz;
                        best.mt = mt; best.nt = nt; best.lds = lds; best.boxes = (unsigned)boxes;
                    }
                }
            }
    if (!found || (cin > 512 && best_cost > 0.93 * gather_cycles(g, cin, ntw))) return false;
    ConvTile& t = best.t;
    const int LX = t.tx + 2, LY = t.ty + 2;
    t.nx = (g.W + t.tx - 1) / t.tx;
    t.ny = (g.H + t.ty - 1) / t.ty;
    t.tv = t.tx * t.ty * t.tz;
    t.pv = (LX * LY * (t.tz + 2) + 15) / 16 * 16;
    t.pu = LX * LY * c8;
    t.row = fast_div(LX * c8); t.c8 = fast_div(c8);
    t.dtx = fast_div(t.tx); t.dty = fast_div(t.ty); t.dnx = block_div(t.nx); t.dny = block_div(t.ny);
    return true;
}

// The plan of a size, searched for once per thread and size while the size keeps its place: the search
// takes 2 to 4 us of the host, which launches of small convolutions in a row wait for (us a launch
// of 8 -> 64 channels, with the search and without: 16^3 5.6 and 4.9, 24^3 6.3 and 4.9).  Null where there is no box.  Threads share nothing.
inline const ConvPlan* kept_plan(const Grid3& g, int cin, int ntw) {
    struct Kept {
        int D, H, W, cin, ntw;
        bool found;
        ConvPlan plan;
    };
    constexpr uint32_t PLACES = 64;  // the network's layers are 23 sizes, 14 KB of a thread's memory
    static thread_local Kept kept[PLACES];
    uint32_t h = 0;
    for (const int v : {g.D, g.H, g.W, cin, ntw}) h = (h ^ (uint32_t)v) * 0x9E3779B1u;
    Kept& k = kept[h >> 26];
    if (k.D != g.D || k.H != g.H || k.W != g.W || k.cin != cin || k.ntw != ntw) {
        k.found = conv_plan(g, cin, ntw, k.plan);
        k.D = g.D; k.H = g.H; k.W = g.W; k.cin = cin; k.ntw = ntw;
    }
    return k.found ? &k.plan : nullptr;
}

}  // namespace mfnn
