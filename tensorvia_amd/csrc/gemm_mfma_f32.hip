// float instantiation of the MFMA GEMM kernels (gemm_mfma_impl.h).
#include "gemm_ms_impl.h"

#include <algorithm>

namespace tvk {
// fp32 matrix cores are 16x slower than the 16-bit ones, so a tile's wasted rows and columns cost
// real time (a 128-row tile computes 128 rows however few are real), and few large tiles leave CUs
// idle that the stream-K split only partly recovers.  Each of the five fp32 tiles is priced as
//   padded MACs / rate / sqrt(min(1, tiles / 128))
// with rates 1.0 (128x128), 0.96 (64x128), 0.94 (128x64), 0.83 (32x128) and 0.77 (128x32): the
// relative speeds on fp32 A[2592, 2048] @ B[2048, 4096] (2,688 / 2,624 / 2,592 padded rows: 353 /
// 363 / 376 / 425 us) and, for 128x32, against 128x64 on shapes of several hundred tiles; the fill
// term was fitted to 50 fp32 shapes (M 20-10000, N 32-11008, K 1000-16384, batch 1, 2, 4, 8 and
// 16) timed on every tile, where the cheapest lands 0.8 % from the fastest on average.  E.g. A[3000, 4096] @
// B[4096, 129]: 128x128 84.5 us, 128x64 60.6 us, 128x32 56.6 us; A[8192, 4096] @ B[4096, 32]:
// 128x64 51.4 us, 128x32 34.8 us; A[300, 4096] @ B[4096, 4096]: 128x128 116.1 us, 64x128 99.7 us.
// A sixth tile, 96x128 (rate 0.984), serves row counts that 96 divides better than 128: on
// A[2592, 2048] @ B[2048, 4096] it computes 2,592 rows instead of 2,688 and ran 341.5-342.7 us
// against 348.5-349.1 us for 128x128 (same box, same process).  Its loaders need A k-contiguous
// (96 rows of an m-contiguous A do not split into whole 16-byte chunks per thread).
namespace {
struct F32Tile {
    int bm, bn;
    double rate;
};
constexpr int kF32TileCount = 6;
constexpr F32Tile kF32Tiles[kF32TileCount] = {{128, 128, 1.0}, {64, 128, 0.96}, {128, 64, 0.94},
                                              {32, 128, 0.83}, {128, 32, 0.77}, {96, 128, 0.984}};

int f32_a_mode_96(const GemmDesc& d) { return pick_mode(d.A, d.M, d.K, d.sa_m, d.sa_k, d.sa_b, d.batch, 4, 96, d.pad_a); }
int f32_b_mode(const GemmDesc& d) { return pick_mode(d.B, d.N, d.K, d.sb_n, d.sb_k, d.sb_b, d.batch, 4, 128, d.pad_b); }

// A 256x256 tile (8 waves of 128x64, one workgroup per CU) reads half the operand bytes per FLOP
// of the 128x128 tile.  It serves shapes whose 256x256 tiles fill whole rounds of the CUs with no
// padded rows or columns: A[4096,4096] @ B[4096,4096] 979.4 against 1,003.9 us, [8192]^3 7,702
// against 7,980 us, [4096,2048] @ [2048,4096] 499.1 against 507.2 us (same box, same process; both
// on the persistent stream-K kernel, before whole rounds took the plain kernel); with
// fewer tiles than CUs the stream-K split it would need measured slower ([2048,8192] @
// [8192,2048], 64 tiles: 533.7 against 518.4 us).
bool f32_whole_rounds_256(const GemmDesc& d) {
    if (d.M % 256 || d.N % 256) return false;
    const int64_t tiles = (int64_t)(d.M / 256) * (d.N / 256) * d.batch;
    const int cus = device_cus();
    return tiles >= cus && tiles % cus == 0;
}

// What these kernels do per us on all CUs ([2592,2048]@[2048,4096]), and the shortest time of a k-tile (32 k)
// in a workgroup, its loads' latency: K = 4096 takes 89 to 96 us on 2 to 64 workgroups of 32x128, whatever M and N.
constexpr double kF32MacsPerUs = 64.4e6, kF32KTileUs = 0.70;

int pick_f32_tile(const GemmDesc& d, bool may_split, double* us) {
    const int bm = f32_b_mode(d);
    const bool t96_ok = f32_a_mode_96(d) == LOAD_KCONTIG && (bm == LOAD_MNCONTIG || bm == LOAD_KCONTIG);
    int best = 0;
    double best_cost = 0;
    for (int i = 0; i < kF32TileCount; ++i) {
        if (i == 5 && !t96_ok) continue;
        const F32Tile& t = kF32Tiles[i];
        const double tm = (double)((d.M + t.bm - 1) / t.bm), tn = (double)((d.N + t.bn - 1) / t.bn);
        const double tiles = (double)d.batch * tm * tn;
        const double fill = tiles >= 128 ? 1.0 : std::sqrt(tiles / 128.0);
        const double cost = tiles * t.bm * t.bn / t.rate / fill;
        if (i == 0 || cost < best_cost) {
            best = i;
            best_cost = cost;
        }
    }
    // The chosen tile's time.
    const F32Tile& t = kF32Tiles[best];
    const int64_t tiles = (int64_t)((d.M + t.bm - 1) / t.bm) * ((d.N + t.bn - 1) / t.bn) * d.batch;
    const int cus = device_cus(), nk = (d.K + 31) / 32;
    const double ktile = t.bm * t.bn * 32 / t.rate / (kF32MacsPerUs / 256); // of a CU's time
    auto step = [&](double tiles_per_cu) { return ktile * tiles_per_cu > kF32KTileUs ? ktile * tiles_per_cu : kF32KTileUs; };
    // A launch with the store of a tile, which the fused epilogue makes longer here: [232,28]@Wt[28,8184] with bias
    // and SiLU 16.4 us, 8.6 on the multi-stage tiles.
    const bool epi = d.bias != nullptr || d.act != TV_ACT_NONE;
    const double mem = ms_mem_us(d), launch = 2.2 + (epi ? 3.0 : 1.3) * t.bm * t.bn / (128 * 128);
    if (may_split && sk_splits(nk, tiles, 2 * cus)) {
        // Whole rounds of two tiles per CU, then the rest in ranges of k-tiles, and the hand-over.
        const int64_t dp = tiles > 2 * cus ? tiles / (2 * cus) * (2 * cus) : 0, iters = (tiles - dp) * nk;
        const int64_t wgs = std::max<int64_t>(1, std::min({iters / 8, (int64_t)2 * cus, 32 * (tiles - dp)}));
        const double k = (double)dp / cus * nk * ktile + (double)iters / wgs * step(std::max(1.0, (double)wgs / cus));
        const double pieces = (double)wgs / (tiles - dp);
        *us = std::max(k, mem) + launch + (pieces > 1.0 ? 9.0 + 0.2 * pieces : 0.0);
    } else {
        *us = std::max(nk * step((double)((tiles + cus - 1) / cus)), mem) + launch + 1.65 * (double)((tiles - 1) / (2 * cus));
    }
    return best;
}

// Calls of few tiles run the multi-stage kernel on 64x64 or 32x64 tiles where that is cheaper: few
// large tiles split over K leave their time in the hand-over.  fp32, us, tiles above -> multi-stage:
// [1024]^3 37.9 -> 23.5, [1001,776]@[776,1004] 28 -> 20.5, [2574,1316]@Wt[1316,320] 40.7 -> 27.9,
// [128,640]@Wt[640,1024] 13.2 -> 8.5, [512]^3 -> 9.3; [2592,2048]@[2048,4096] 343 against 347 there.
// Both prices (as in gemm_ms_impl.h, 32 k per k-tile; the matrix cores' time bounds these) are fitted to
// 1,145 random fp32 calls (1 to 60,000 rows, 4 to 125,000 k) timed on the tiles above and on each of these whole
// and split: 2 % from the fastest on average.  Where a call is bound by its output, or is one or two k-tiles on
// large tiles, the tiles above win (us, there / here): [11,32]@Wt[32,26480] 3.8 / 4.9, [96,64]@[64,26512] 7.8 /
// 11.1, [25008,8]@[8,4] 4.1 / 5.9, [43376,32]@Wt[32,16] 5.4 / 7.0, [34704,304]@Wt[304,31] 17.2 / 21.2; but
// [504,4]@Wt[4,164] 5.2 / 4.0.
constexpr MsTile kF32MsTiles[2] = {{32, 64, 3, 2.1, 2.5, 1.0, 0.47, 0.91, 3.0, 0.25}, {64, 64, 3, 2.9, 3.4, 1.0, 0.63, 1.56, 3.0, 0.25}};

int run_f32_ms(const GemmDesc& d, hipStream_t stream, bool may_alloc, double other_us) { // 1: not cheaper
    const int am = pick_mode(d.A, d.M, d.K, d.sa_m, d.sa_k, d.sa_b, d.batch, 4, 128, d.pad_a), bm = f32_b_mode(d);
    if (am == LOAD_GENERIC || bm == LOAD_GENERIC) return 1;
    const bool ok[2] = {am == LOAD_KCONTIG, true};
    // N-contiguous B is read in pieces of 256 bytes, half of what the 128-column tiles read: streamed from memory
    // that costs about a tenth ([25,7616]@[7616,12640] 82 to 94 us here, 78 on tiles of 32x128).
    const MsPlan plan = ms_plan(d, (d.K + 31) / 32, kF32MsTiles, ok, 2, may_alloc, bm == LOAD_MNCONTIG ? 1.1 : 1.0);
    // Above one chunk of k this kernel's sums are the more accurate ones (2e-7 relative against 2e-7 to 6e-7, growing
    // with K): it is taken for up to a tenth more, at most 1 us.
    if (plan.us >= other_us + (d.K > 128 ? std::min(0.1 * other_us, 1.0) : 0.0)) return 1;
#define TV_MS(TILE_, BM_, WM_, WN_, NST_, A_, B_) \
    if (plan.tile == TILE_ && am == A_ && bm == B_) return run_ms_cfg<GemmCfg<float, BM_, 64, WM_, WN_, A_, B_>, NST_>(d, stream, plan);
    TV_MS(0, 32, 1, 4, 4, LOAD_KCONTIG, LOAD_KCONTIG)
    TV_MS(0, 32, 1, 4, 4, LOAD_KCONTIG, LOAD_MNCONTIG)
    TV_MS(1, 64, 2, 2, 3, LOAD_KCONTIG, LOAD_KCONTIG)
    TV_MS(1, 64, 2, 2, 3, LOAD_KCONTIG, LOAD_MNCONTIG)
    TV_MS(1, 64, 2, 2, 3, LOAD_MNCONTIG, LOAD_KCONTIG)
    TV_MS(1, 64, 2, 2, 3, LOAD_MNCONTIG, LOAD_MNCONTIG)
#undef TV_MS
    return 1;
}
} // namespace

int launch_gemm_mfma_f32(const GemmDesc& d, hipStream_t stream, bool may_alloc) {
    double us = 0;
    const int tile = pick_f32_tile(d, may_alloc, &us);
    const int rc = run_f32_ms(d, stream, may_alloc, us);
    if (rc == TV_E_NOMEM) return launch_gemm_mfma_f32(d, stream, false);
    if (rc != 1) return rc;
    switch (tile) {
        case 0:
            if (f32_whole_rounds_256(d)) return run_modes<float, 256, 256, 2, 4>(d, stream, 8, may_alloc);
            return run_modes<float, 128, 128, 2, 2>(d, stream, 8, may_alloc);
        case 1: return run_modes<float, 64, 128, 2, 2>(d, stream, 8, may_alloc);
        case 2: return run_modes<float, 128, 64, 2, 2>(d, stream, 8, may_alloc);
        case 3: return run_modes<float, 32, 128, 1, 4>(d, stream, 8, may_alloc);
        case 4: return run_modes<float, 128, 32, 4, 1>(d, stream, 8, may_alloc);
        default:
            if (f32_b_mode(d) == LOAD_MNCONTIG)
                return run_cfg<GemmCfg<float, 96, 128, 2, 2, LOAD_KCONTIG, LOAD_MNCONTIG>>(d, stream, 8, may_alloc);
            return run_cfg<GemmCfg<float, 96, 128, 2, 2, LOAD_KCONTIG, LOAD_KCONTIG>>(d, stream, 8, may_alloc);
    }
}
} // namespace tvk
