// Multi-stage direct-load GEMM for launches of few tiles (fp32, 16-bit and int8 inputs, both operands
// in a vector layout).
//
// With at most about one tile per CU a workgroup has the CU to itself, and what bounds it is the
// latency of its own loads: two LDS stages keep one k-tile in flight, so every k-tile costs the round
// trip to L2 or HBM, about 1 us, whatever its work (bf16 [333,4096]@[4096,11008], 258 tiles of
// 128x128: 62 us for 64 k-tiles whose MFMAs take 14 us).  Here NST stages (4 of 32 KB for a 128x128
// tile) keep NST - 1 k-tiles in flight, which is what LDS is large enough for at this occupancy.
//  * The operands' layouts in LDS, the direct loads and the fragment reads are DmaOperand's
//    (gemm_dma_impl.h).
//  * One barrier per k-tile t: wait until k-tile t + 1 has landed (vmcnt retires in issue order),
//    barrier (it is visible to every wave, and every wave is done with the stage of t - 1), issue
//    the loads of k-tile t + NST - 1 into that stage.  Then the MFMAs of k-group 0 with the reads of
//    k-group 1's fragments between them, and those of k-group 1 with the reads of k-tile t + 1's
//    k-group 0: LDS, which delivers a wave tile's fragments no faster than the matrix cores use them,
//    works while they do.
//  * Smaller tiles (down to 32x64 with 4 waves) where the large ones leave CUs idle.
//  * Rotation: where one operand is streamed once in rows of k (K-contiguous, each tile its own rows)
//    and the other is small enough to stay in the XCDs' L2s, tile i starts its k-loop at k-tile
//    i mod n and wraps round.  Started together at k = 0, all tiles read the same 128 bytes of rows
//    whose pitch is a large power of two, which fall on few of the memory channels: bf16
//    [65536,2048]@[2048,128] 73.7 -> 53.6 us rotated (4.9 -> 5.6 TB/s of reads; 256x128 tiles).  Tiles
//    that share a large operand must stay in step instead ([1024,4096]@[4096,4096] 41.1 -> 45.6).
//  * The schedule is gemm_mfma_sk_kernel's: a tile per workgroup, or all tiles split over K in equal
//    ranges of (tile, k-tile) iterations, partial sums through slots, summed in segment order by the
//    segment that arrives last.  No workgroup waits for another.
#pragma once
#include "gemm_dma_impl.h"

#include <utility>

namespace tvk {

template <class C, int NST> constexpr int ms_lds_bytes() {
    return NST * (DmaOperand<C::AMODE, C::BM, C::THREADS, C::ES>::BYTES + DmaOperand<C::BMODE, C::BN, C::THREADS, C::ES>::BYTES);
}

struct MsArgs {
    int64_t iters; // split: tiles x k-tiles; 0: workgroup w computes tile w
    int nk;        // k-tiles per tile
    int rot;       // 1: tiles start their k-loops rotated by their tile row
    int* cnt;      // [tiles] arrival counters, zero between launches
    char* slots;   // [2 x workgroups][slot bytes]
};

// k-tiles [kt0, kt1) of one output tile, starting `rot` k-tiles into the range and wrapping round, into
// acc (zeroed by the caller); 0 <= rot < kt1 - kt0.  Entered with the LDS free (after a workgroup
// barrier), left with every load landed.
template <class C, int NST>
__device__ __attribute__((always_inline)) inline void ms_tile_kloop(const GemmDesc& d, char* L, int b, int m0, int n0, int kt0,
                                                                    int kt1, int rot, typename Mfma<typename C::T>::Acc (&acc)[C::FM][C::FN]) {
    using Op = Mfma<typename C::T>;
    constexpr int ES = C::ES;
    using LA = DmaOperand<C::AMODE, C::BM, C::THREADS, ES>;
    using LB = DmaOperand<C::BMODE, C::BN, C::THREADS, ES>;
    constexpr int NDMA = LA::PER_WAVE + LB::PER_WAVE;
    static_assert(NST >= 3 && (NST - 2) * NDMA < 64, "stages; vmcnt range");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / C::WAVES_N, wn = wave % C::WAVES_N;
    const unsigned LA0 = (unsigned)(uintptr_t)(lds_void*)L;
    const unsigned LB0 = LA0 + NST * LA::BYTES;
    const int K_eff = min(d.K, kt1 * C::BK); // loads past the range return zeros

    LA la;
    la.base = static_cast<const char*>(d.A) + ((int64_t)b * d.sa_b + (int64_t)m0 * d.sa_m) * ES;
    la.s_r = d.sa_m; la.s_k = d.sa_k; la.rows_valid = d.M - m0; la.K = K_eff;
    LB lb;
    lb.base = static_cast<const char*>(d.B) + ((int64_t)b * d.sb_b + (int64_t)n0 * d.sb_n) * ES;
    lb.s_r = d.sb_n; lb.s_k = d.sb_k; lb.rows_valid = d.N - n0; lb.K = K_eff;
    la.init(wave, lane);
    lb.init(wave, lane);
    la.xinit(LA0, lane, wm * C::WM);
    lb.xinit(LB0, lane, wn * C::WN);

    auto k_of = [&](int kt) { // past the range: zeros, from the loaders' K
        if (kt < kt1) {
            kt += rot;
            kt = kt < kt1 ? kt : kt - (kt1 - kt0);
        }
        return kt * C::BK;
    };
    auto issue = [&](int kt, int st) {
        la.issue(L + st * LA::BYTES, wave, k_of(kt));
        lb.issue(L + NST * LA::BYTES + st * LB::BYTES, wave, k_of(kt));
    };
    // A fragments: one set, each reloaded with the next k-group's right after its row of MFMAs; B
    // fragments: one set per k-group.
    u32x4 fa[C::FM], fb[2][C::FN];
    // MFMAs of one k-group (B set `cur`), reading k-group kg of the k-tile at xa / xb into the other set;
    // after(i) runs behind row i's MFMAs.
    auto kgroup = [&](int cur, unsigned xa, unsigned xb, int kg, const auto& after) {
#pragma unroll
        for (int i = 0; i < C::FM; ++i) {
#pragma unroll
            for (int j = 0; j < C::FN; ++j) Op::run(fb[cur][j], fa[i], acc[i][j]);
            after(i);
            fa[i] = LA::frag_from(xa, 0, kg, i);
#pragma unroll
            for (int j = i * C::FN / C::FM; j < (i + 1) * C::FN / C::FM; ++j) fb[cur ^ 1][j] = LB::frag_from(xb, 0, kg, j);
        }
        // Each row's MFMAs, then the reads that follow that row.
        [&]<int... I>(std::integer_sequence<int, I...>) {
            ((__builtin_amdgcn_sched_group_barrier(SG_MFMA, C::FN * Op::kInstr, 0),
              __builtin_amdgcn_sched_group_barrier(
                  SG_DS_READ, LA::kFragReads + ((I + 1) * C::FN / C::FM - I * C::FN / C::FM) * LB::kFragReads, 0)),
             ...);
        }(std::make_integer_sequence<int, C::FM>());
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int s = 0; s < NST - 1; ++s) issue(kt0 + s, s);
    wait_vmcnt<(NST - 2) * NDMA>();
    dma_barrier();
#pragma unroll
    for (int j = 0; j < C::FN; ++j) fb[0][j] = LB::frag_from(lb.xf, 0, 0, j);
#pragma unroll
    for (int i = 0; i < C::FM; ++i) fa[i] = LA::frag_from(la.xf, 0, 0, i);
    int st = 0;
    auto ktile = [&](int kt) {
        const int fs = st == 0 ? NST - 1 : st - 1; // the stage freed last step
        const unsigned xa = la.xf + (unsigned)(st * LA::BYTES), xb = lb.xf + (unsigned)(st * LB::BYTES);
        // The loads of k-tile t + NST - 1.  On the small 16-bit and int8 tiles they go out between the
        // rows of MFMAs, beside which their issue (about 40 cycles each) runs: bf16
        // [128,4096]@Wt[4096,4096] on 64x64 tiles 20.4 -> 18.8 us.  On the large tiles, whose second wave
        // per SIMD covers it, and in fp32 all at once (128x128: bf16 [1024,4096]@[4096,4096] 41.1 us, 42.8
        // between the rows; fp32 [1024]^3 23.5, 26.2).
        if constexpr (ES <= 2 && C::FM * C::FN <= 4) {
            const int k2 = k_of(kt + NST - 1);
            const __amdgpu_buffer_rsrc_t ra = la.rsrc(k2), rb = lb.rsrc(k2);
            const unsigned sa = LA0 + (unsigned)(fs * LA::BYTES), sb = LB0 + (unsigned)(fs * LB::BYTES);
            wait_vmcnt<(NST - 3) * NDMA>();
            dma_barrier();
            kgroup(0, xa, xb, 1, [&](int i) {
#pragma unroll
                for (int u = i * NDMA / C::FM; u < (i + 1) * NDMA / C::FM; ++u) {
                    if (u < LA::PER_WAVE) la.issue_one(u, ra, sa, wave, k2);
                    else lb.issue_one(u - LA::PER_WAVE, rb, sb, wave, k2);
                }
            });
        } else {
            wait_vmcnt<(NST - 3) * NDMA>();
            dma_barrier();
            issue(kt + NST - 1, fs);
            kgroup(0, xa, xb, 1, [](int) {});
        }
        st = st + 1 == NST ? 0 : st + 1;
        kgroup(1, la.xf + (unsigned)(st * LA::BYTES), lb.xf + (unsigned)(st * LB::BYTES), 0, [](int) {});
    };
    // fp32 results in chunks of kChunk k-tiles, each summed by itself and then added: rounding grows
    // with the chunk's length and the chunk count, not with K (fp32 [1001,777]@[777,1003]: 2.6e-7
    // relative error against 64 bits, 5e-7 in one chain).  The small tiles have the registers for it.
    // 16-bit results round far above that, and their loop stays the plain one (5 % faster).
    constexpr int kChunk = ES == 4 ? 4 : 16;
    constexpr bool kMayChunk = !__is_same(typename C::T, int8_t) && C::FM * C::FN <= 4;
    if (kMayChunk && d.dtype_c == TV_FLOAT32) {
        typename Op::Acc sum[C::FM][C::FN];
        for (int c0 = kt0; c0 < kt1; c0 += kChunk) {
            const int c1 = min(c0 + kChunk, kt1);
            for (int kt = c0; kt < c1; ++kt) ktile(kt);
#pragma unroll
            for (int i = 0; i < C::FM; ++i)
#pragma unroll
                for (int j = 0; j < C::FN; ++j) {
                    sum[i][j] = c0 == kt0 ? acc[i][j] : sum[i][j] + acc[i][j];
                    acc[i][j] = typename Op::Acc{0, 0, 0, 0};
                }
        }
#pragma unroll
        for (int i = 0; i < C::FM; ++i)
#pragma unroll
            for (int j = 0; j < C::FN; ++j) acc[i][j] = sum[i][j];
    } else {
        for (int kt = kt0; kt < kt1; ++kt) ktile(kt);
    }
    wait_vmcnt<0>();
}

template <class C, int NST, bool FUSED>
__global__ __attribute__((amdgpu_flat_work_group_size(C::THREADS, C::THREADS), amdgpu_waves_per_eu(2)))
void gemm_ms_kernel(GemmDesc d, int tiles_m, int tiles_n, int group_m, int c_vec, MsArgs ms) {
    using Acc = typename Mfma<typename C::T>::Acc;
    constexpr int SLOT = sk_slot_bytes<C>();
    __shared__ __attribute__((aligned(1024))) char L[ms_lds_bytes<C, NST>()];
    int* const last_flag = reinterpret_cast<int*>(L); // used between a k-loop and the store, when L is free
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int G = gridDim.x;
    int w = blockIdx.x;
    if ((G & 7) == 0) w = (w & 7) * (G >> 3) + (w >> 3); // consecutive ids on one XCD
    const int nk = ms.nk;
    const int64_t I = ms.iters;
    // Workgroup w's range of iterations; unsplit, those of tile w.
    const int64_t it_begin = I > 0 ? (int64_t)w * I / G : (int64_t)w * nk;
    const int64_t it_end = I > 0 ? (int64_t)(w + 1) * I / G : it_begin + nk;
    // The workgroup whose range holds iteration it: the largest v with floor(v * I / G) <= it.
    auto owner = [&](int64_t it) { return (int)(((it + 1) * G - 1) / I); };
    auto slot_rsrc = [&](int slot) { return make_rsrc(ms.slots + (int64_t)slot * SLOT, SLOT); };
    for (int64_t it = it_begin; it < it_end;) {
        const int tile = (int)(it / nk);
        const int kt0 = (int)(it - (int64_t)tile * nk);
        const int kt1 = (int)min((int64_t)nk, kt0 + (it_end - it));
        it += kt1 - kt0;
        int b, tm, tn;
        mfma_tile_of(tile, tiles_m, tiles_n, group_m, b, tm, tn);
        const int m0 = tm * C::BM, n0 = tn * C::BN;
        const int rot = ms.rot ? (int)(((int64_t)b * tiles_m + tm) % (kt1 - kt0)) : 0;
        Acc acc[C::FM][C::FN];
#pragma unroll
        for (int i = 0; i < C::FM; ++i)
#pragma unroll
            for (int j = 0; j < C::FN; ++j) acc[i][j] = Acc{0, 0, 0, 0};
        lds_barrier(); // the previous segment's epilogue is done with the LDS
        ms_tile_kloop<C, NST>(d, L, b, m0, n0, kt0, kt1, rot, acc);
        if (kt0 != 0 || kt1 != nk) {
            const int64_t t0 = (int64_t)tile * nk;
            const int first = owner(t0), last = owner(t0 + nk - 1);
            {
                const __amdgpu_buffer_rsrc_t r = slot_rsrc(w == first ? 2 * w + 1 : 2 * w);
#pragma unroll
                for (int i = 0; i < C::FM; ++i)
#pragma unroll
                    for (int j = 0; j < C::FN; ++j)
                        slot_store16(r, (((wave * C::FM + i) * C::FN + j) * 64 + lane) * 16, acc[i][j]);
            }
            lds_barrier(); // every wave is done with the k-loop's LDS
            publish_and_count(ms.cnt + tile, last - first + 1, last_flag);
            if (!*last_flag) continue;
            // Sum the segments' slots in segment order (this workgroup's own included), the loads of U
            // segments in flight at a time (past the last: out of range, zeros).
            constexpr int U = C::FM * C::FN <= 4 ? 4 : C::FM * C::FN <= 8 ? 2 : 1;
#pragma unroll
            for (int i = 0; i < C::FM; ++i)
#pragma unroll
                for (int j = 0; j < C::FN; ++j) acc[i][j] = Acc{0, 0, 0, 0};
            for (int v = first; v <= last; v += U) {
                Acc p[U][C::FM][C::FN];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const __amdgpu_buffer_rsrc_t r = slot_rsrc(v + u == first ? 2 * (v + u) + 1 : 2 * min(v + u, last));
#pragma unroll
                    for (int i = 0; i < C::FM; ++i)
#pragma unroll
                        for (int j = 0; j < C::FN; ++j) {
                            const int off = (((wave * C::FM + i) * C::FN + j) * 64 + lane) * 16;
                            p[u][i][j] = slot_load16<Acc>(r, v + u <= last ? off : (int)kOOB);
                        }
                }
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int i = 0; i < C::FM; ++i)
#pragma unroll
                        for (int j = 0; j < C::FN; ++j) acc[i][j] = acc[i][j] + p[u][i][j];
            }
            slot_count_reset(ms.cnt + tile);
        }
        dma_tile_store<C, FUSED>(d, L, b, m0, n0, c_vec, acc);
    }
}

// ---------------------------------------------------------------------------------------------
// Host side: the tile and the split of one call.

// A tile as the plan prices it, in us: `fixed` for a launch (first loads, the store), `round` more for
// each further round of workgroups, `share` for a CU's second and third workgroup, t1 per k-tile for a workgroup that has its CU to itself and tr
// when `occ` of them share it (all CUs busy); a split (where it can: s0 >= 0) costs s0 plus s1 per
// segment of a tile (slots written, the hand-over, the last segment's sums).
struct MsTile {
    int bm, bn, occ;
    double fixed, round, share, t1, tr, s0, s1;
};
struct MsPlan {
    int tile = -1; // index into the tile list
    int64_t wgs = 0;
    bool split = false;
    double us = 0;
};
constexpr double kMsBytesPerUs = 5.0e6; // what the largest streams of these calls reach

// The least time of d's operands and result in memory, each read or written once.
static double ms_mem_us(const GemmDesc& d) {
    const double b = d.batch;
    return (((d.sa_b ? b : 1) * d.M + (d.sb_b ? b : 1) * d.N) * d.K * (double)dtype_size(d.dtype_a) +
            b * d.M * d.N * (double)dtype_size(d.dtype_c)) / kMsBytesPerUs;
}

// The cheapest of `tiles` (those with ok set) for nk k-tiles of d; none where no grid of them fits.
static MsPlan ms_plan(const GemmDesc& d, int nk, const MsTile* tiles, const bool* ok, int n, bool may_split, double mem_scale = 1.0) {
    const int cus = device_cus();
    const double mem = ms_mem_us(d) * mem_scale;
    MsPlan best;
    for (int i = 0; i < n; ++i) {
        if (!ok[i]) continue;
        const MsTile& t = tiles[i];
        const int64_t nt = (int64_t)((d.M + t.bm - 1) / t.bm) * ((d.N + t.bn - 1) / t.bn) * d.batch;
        const int64_t slots = (int64_t)cus * t.occ;
        if (nt * (t.bm * t.bn <= 64 * 64 ? 256 : 512) > 0xFFFFFFFFll) continue; // a grid holds fewer than 2^32 threads
        // us per k-tile with w workgroups in flight.  Unsplit plans count a handful of tiles more than CUs as half a
        // second workgroup on the two-stage tile: bf16 [333,4096]@[4096,11008], 258 tiles, 56 us, 512 of them 77.
        auto step = [&](int64_t w) {
            const double load = (double)((w + cus - 1) / cus - 1);
            if (t.occ == 1 || load <= 0) return t.t1;
            const bool handful = !may_split && t.s0 < 0 && w * 16 <= (int64_t)cus * 17;
            return t.t1 + (t.tr - t.t1) * (handful ? 0.5 : load) / (t.occ - 1);
        };
        auto offer = [&](int64_t wgs, bool split, double k_us, double more) {
            const double us = t.fixed + (k_us > mem ? k_us : mem) + more;
            if (best.tile < 0 || us < best.us) best = MsPlan{i, wgs, split, us};
        };
        const int64_t full = nt / slots, rest = nt % slots;
        // A CU's second and third workgroup start beside the first, not for nothing (fp16
        // [13][128,512]@[512,928] on 390 tiles of 64x64 11.2 us, 9.4 on 128x128).
        const double start = t.occ == 1 || nt <= cus ? 0.0 : t.share * (double)((nt < slots ? (nt + cus - 1) / cus : t.occ) - 1);
        offer(nt, false, nk * (full * step(slots) + (rest ? step(rest) : 0)), start + t.round * (double)(full + (rest != 0) - 1));
        if (!may_split || t.s0 < 0 || nt > 0x3FFFFFFF / (nk > 0 ? nk : 1)) continue;
        for (int s = 2; s <= 64 && nt * s <= slots && nk >= 2 * s; s += s < 8 ? 1 : s / 4)
            offer(nt * s, true, (double)nk / s * step(nt * s), t.s0 + t.s1 * s);
        // A range of equal length for every workgroup that the CUs hold: most tiles in two pieces.  Not on
        // 32x64 tiles, three per CU, which read the operands from L2 too often (fp32 [224,59008]@Wt[59008,462] 181 us,
        // 136 on 64x64).
        if (t.bm > 32 && nt * nk >= 4 * slots && rest != 0)
            offer(slots, true, (double)nt * nk / slots * step(slots), t.s0 + t.s1 * (2 + (double)slots / nt) + t.round * (double)(full + 1));
    }
    return best;
}

// Whether the tiles stream A in rows of k while B stays in L2 (see the rotation above): B within half
// of an XCD's 4 MB, and few tile columns.  Rotating by tile column where B is streamed in rows of k
// changed nothing (fp16 [48,4096]@Wt[4096,11008] 21.8 us either way) and is not done.
static bool ms_rotation(const GemmDesc& d, int es, int am, int64_t tiles_m, int64_t tiles_n) {
    return am == LOAD_KCONTIG && (int64_t)d.K * d.N * es <= (int64_t)2 << 20 && tiles_m >= 4 * tiles_n;
}

// TV_E_NOMEM: no room for the slots of a split plan; the caller plans again without a split (the tile
// chosen for a split may be a poor one whole: bf16 [333,4096]@[4096,11008], 258 tiles of 128x128 that
// fill one CU each, are two rounds of 64 k-tiles).
template <class C, int NST>
static int run_ms_cfg(const GemmDesc& d, hipStream_t stream, const MsPlan& plan) {
    constexpr int kGroupM = 8;
    const int64_t tiles_m = (d.M + C::BM - 1) / C::BM, tiles_n = (d.N + C::BN - 1) / C::BN;
    const int64_t nt = tiles_m * tiles_n * d.batch;
    if (nt <= 0) return 0;
    if (nt > 0x7FFFFFFF) return TV_E_SHAPE;
    const bool epi = d.bias != nullptr || d.act != TV_ACT_NONE;
    if (epi && d.sc_n != 1) return TV_E_UNSUPPORTED; // the fused store writes rows of C
    MsArgs ms;
    ms.nk = (d.K + C::BK - 1) / C::BK;
    ms.iters = 0;
    ms.rot = ms_rotation(d, C::ES, C::AMODE, tiles_m * d.batch, tiles_n);
    ms.cnt = nullptr;
    ms.slots = nullptr;
    int64_t G = nt;
    if (plan.split) {
        const int rc = gemm_sk_workspace(stream, (size_t)nt, (size_t)2 * plan.wgs * sk_slot_bytes<C>(), &ms.cnt, &ms.slots);
        if (rc) return rc;
        G = plan.wgs;
        ms.iters = nt * ms.nk;
    }
    const int c_vec = c_store_mode(d);
    if constexpr (!__is_same(typename C::T, int8_t))
        if (epi) {
            hipLaunchKernelGGL((gemm_ms_kernel<C, NST, true>), dim3((unsigned)G), dim3(C::THREADS), 0, stream, d, (int)tiles_m,
                               (int)tiles_n, kGroupM, c_vec, ms);
            return hipGetLastError();
        }
    hipLaunchKernelGGL((gemm_ms_kernel<C, NST, false>), dim3((unsigned)G), dim3(C::THREADS), 0, stream, d, (int)tiles_m, (int)tiles_n,
                       kGroupM, c_vec, ms);
    return hipGetLastError();
}

// Tiles of the 16-bit and int8 inputs.  Prices: bf16 with K of 64 to 4096, from about 30 shapes of 16 to
// 16128 rows timed on every tile and split (e.g. bf16 [64,3712]@Wt[3712,1216] 64x64: 17.2 us whole, 9.7
// in 4 or 8 pieces, 128x128: 27.3 whole; [600,4096]@[4096,4096] 128x128 38.2, 256x128 55.7; [2048,4096]
// @[4096,4096] 256x128 63.1, 128x128 77.4).  int8 k-tiles hold twice the k for the same bytes and
// matrix-core cycles.  The last two are the kernels of gemm_dma_impl.h: 128x128 tiles with two stages,
// two workgroups per CU, which start faster (bf16 [8][512,96]@Kt[96,512] 5.0 us against 6.2 here), and
// 256x256 tiles (bf16 [4096]^3 98 us).
enum { MS_32x64, MS_64x64, MS_64x128, MS_128x128, MS_256x128, MS_DMA_128, MS_DMA_256, MS_TILES };
constexpr MsTile kMsTiles[MS_TILES] = {{32, 64, 3, 3.5, 2.0, 1.5, 0.25, 0.43, 3.0, 0.25},  {64, 64, 2, 4.8, 2.6, 1.5, 0.25, 0.43, 3.0, 0.25},
                                       {64, 128, 1, 5.0, 3.0, 0.0, 0.42, 0.42, 4.0, 0.35}, {128, 128, 1, 5.0, 4.0, 0.0, 0.58, 0.58, 5.0, 0.6},
                                       {256, 128, 1, 6.5, 5.5, 0.0, 0.9, 0.9, 8.0, 1.2},   {128, 128, 2, 3.8, 2.5, 0.0, 0.67, 0.95, -1, 0},
                                       {256, 256, 1, 9.0, 7.0, 0.0, 1.3, 1.3, -1, 0}};

// Runs d on the cheapest tile; 1 if that is the 256x256 one, TV_E_NOMEM as run_ms_cfg.  am / bm: the operands' (vector) load modes.
template <typename T>
static int run_modes_ms(const GemmDesc& d, hipStream_t stream, int group_m, int am, int bm, bool may_alloc) {
    constexpr bool kI8 = __is_same(T, int8_t);
    const int nk = (d.K + 128 / (int)sizeof(T) - 1) / (128 / (int)sizeof(T));
    // Layouts: 32 rows K-contiguous only; 64 rows M/N-contiguous at 16 bits only (DmaOperand).
    const bool r64a = am == LOAD_KCONTIG || !kI8, r64b = bm == LOAD_KCONTIG || !kI8;
    // Two shapes outside the prices, measured on 507 calls of up to 131,072 rows or columns, K of 64 to 8192:
    //  * Tall: A streamed in rows of whole 4 KB by tiles of one column (N above 64, in batches from 96), at least
    //    one 256x128 tile per CU, up to 512 MB of A: 256x128, rotated.  us, 256x128 rotated / 128x128: bf16
    //    [65536,2048]@[2048,128] 42.2 / 49.6, [131072,2048]@[2048,72] 114 / 132, [65536,4096]@[4096,128] 107 / 128,
    //    32 batches of [2048,2048] with a [2048,128] each 53.6 / 58.5.  Outside: 3072 k (6 KB) 86.5 / 83.9 at N = 96, 16 batches of
    //    [4096,2048] with 80 columns each 51.0 / 45.2, 50,000 rows (0.77 tiles per CU) 43.3 / 35.0, [131072,4096]
    //    (1 GB) 213 / 200.
    //  * Strip: one row or column of 256x256 tiles, where 128x128 tiles would be more than the CUs hold and read the
    //    large operand twice: 256x256.  us, 256x256 / 128x128: bf16 [224,384]@[384,49184] 15.3 / 23.0, [256,1024]@
    //    [1024,40960] 25.9 / 29.5, [131072,1152]@[1152,256] 81.8 / 108, int8 [49152,6144]@[6144,256] 82.8 / 112, 256
    //    batches of [160,1024]@[1024,160] 33.0 / 35.0; not where the second round is less than half full
    //    ([76512,880]@[880,176], 299 tiles: 59.2 / 46.9), nor for little more than 128 columns ([131072,256]@[256,136]
    //    40.2 / 30.4) or few k-tiles of a tall one (56 batches of [2960,136]@[136,200] 66.1 / 40.8).
    const int64_t cus = device_cus();
    const int64_t tall_m = ((int64_t)d.M + 255) / 256 * d.batch, tall_n = (d.N + 127) / 128;
    const bool tall = d.N > (d.batch > 1 ? 95 : 64) && d.N <= 128 && nk >= 8 && d.sa_m * (int64_t)sizeof(T) % 4096 == 0 && tall_m >= cus &&
                      (int64_t)d.M * d.batch * d.sa_m * (int64_t)sizeof(T) <= (int64_t)512 << 20 && ms_rotation(d, (int)sizeof(T), am, tall_m, tall_n);
    const int64_t nt128 = ((int64_t)d.M + 127) / 128 * tall_n * d.batch, nt256 = tall_m * ((d.N + 255) / 256);
    const bool strip = d.M >= 144 && d.N >= 160 && (d.M <= 256 || (d.N <= 256 && nk >= 8)) && nt128 > 2 * cus &&
                       (nt256 <= cus || nt256 * 4 >= (nt256 + cus - 1) / cus * cus * 3);
    if (strip) return 1;
    // 32x64 tiles up to one per CU: more of them read B from L2 too often (fp16 [3][128,448]@[448,2744],
    // 516 tiles, 12.7 us; 9.2 on 64x64 or 128x128).
    const bool few32 = ((int64_t)d.M + 31) / 32 * (((int64_t)d.N + 63) / 64) * d.batch <= device_cus();
    const bool ok[MS_TILES] = {am == LOAD_KCONTIG && r64b && few32, r64a && r64b, kI8 && am == LOAD_KCONTIG && !r64b, true, true, true, true};
    MsPlan plan = ms_plan(d, nk, kMsTiles, ok, MS_TILES, may_alloc);
    if (tall) plan = MsPlan{MS_256x128, 0, false, 0};
    if (plan.tile == MS_DMA_256) return 1;
#define TV_DMA(A_, B_) \
    if (plan.tile == MS_DMA_128 && am == A_ && bm == B_) return run_dma_cfg<GemmCfg<T, 128, 128, 2, 4, A_, B_>>(d, stream, group_m);
    TV_DMA(LOAD_KCONTIG, LOAD_MNCONTIG)
    TV_DMA(LOAD_KCONTIG, LOAD_KCONTIG)
    TV_DMA(LOAD_MNCONTIG, LOAD_MNCONTIG)
    TV_DMA(LOAD_MNCONTIG, LOAD_KCONTIG)
#undef TV_DMA
#define TV_MS(TILE_, BM_, BN_, WM_, WN_, NST_, A_, B_) \
    if (plan.tile == TILE_ && am == A_ && bm == B_) return run_ms_cfg<GemmCfg<T, BM_, BN_, WM_, WN_, A_, B_>, NST_>(d, stream, plan);
#define TV_MS_B(TILE_, BM_, BN_, WM_, WN_, NST_, A_) \
    TV_MS(TILE_, BM_, BN_, WM_, WN_, NST_, A_, LOAD_KCONTIG) TV_MS(TILE_, BM_, BN_, WM_, WN_, NST_, A_, LOAD_MNCONTIG)
    if constexpr (kI8) {
        TV_MS(MS_32x64, 32, 64, 1, 4, 4, LOAD_KCONTIG, LOAD_KCONTIG)
        TV_MS(MS_64x64, 64, 64, 2, 2, 5, LOAD_KCONTIG, LOAD_KCONTIG)
        TV_MS(MS_64x128, 64, 128, 2, 4, 5, LOAD_KCONTIG, LOAD_MNCONTIG)
    } else {
        TV_MS_B(MS_32x64, 32, 64, 1, 4, 4, LOAD_KCONTIG)
        TV_MS_B(MS_64x64, 64, 64, 2, 2, 5, LOAD_KCONTIG)
        TV_MS_B(MS_64x64, 64, 64, 2, 2, 5, LOAD_MNCONTIG)
    }
    TV_MS_B(MS_128x128, 128, 128, 2, 4, 4, LOAD_KCONTIG)
    TV_MS_B(MS_128x128, 128, 128, 2, 4, 4, LOAD_MNCONTIG)
    TV_MS_B(MS_256x128, 256, 128, 4, 2, 3, LOAD_KCONTIG)
    TV_MS_B(MS_256x128, 256, 128, 4, 2, 3, LOAD_MNCONTIG)
#undef TV_MS_B
#undef TV_MS
    return 1;
}

// 16-bit / int8 inputs: small K, then this file's kernel or 256x256 tiles for the vector layouts,
// gemm_mfma_kernel otherwise.
template <typename T>
static int run_modes_dma(const GemmDesc& d, hipStream_t stream, int group_m, bool may_alloc) {
    const int es = (int)sizeof(T);
    const int am = pick_mode(d.A, d.M, d.K, d.sa_m, d.sa_k, d.sa_b, d.batch, es, 256, d.pad_a);
    const int bm = pick_mode(d.B, d.N, d.K, d.sb_n, d.sb_k, d.sb_b, d.batch, es, 256, d.pad_b);
    if (am == LOAD_GENERIC || bm == LOAD_GENERIC) return run_modes<T, 256, 256, 2, 4>(d, stream, group_m, may_alloc);
    // The small-K kernels have no fused epilogue (their staging area holds the output type only).
    const bool epi = d.bias != nullptr || d.act != TV_ACT_NONE;
    const bool smallk = !epi && smallk_ok(d, es, 256, 256);
    if (!smallk) {
        int rc = run_modes_ms<T>(d, stream, group_m, am, bm, may_alloc);
        if (rc == TV_E_NOMEM) rc = run_modes_ms<T>(d, stream, group_m, am, bm, false);
        if (rc != 1) return rc;
    }
#define TV_CASE(A_, B_)                                                                         \
    if (am == A_ && bm == B_) {                                                                 \
        if (smallk) {                                                                           \
            if constexpr (sizeof(T) == 2) {                                                     \
                const int rc = run_smallk_pipe_cfg<GemmCfg<T, 128, 128, 2, 4, A_, B_>>(d, stream); \
                if (rc != 1) return rc;                                                         \
            }                                                                                   \
            return run_smallk_cfg<GemmCfg<T, 256, 256, 2, 4, A_, B_>>(d, stream);               \
        }                                                                                       \
        return run_dma_cfg<GemmCfg<T, 256, 256, 2, 4, A_, B_>>(d, stream, group_m);             \
    }
    TV_CASE(LOAD_KCONTIG, LOAD_MNCONTIG)
    TV_CASE(LOAD_KCONTIG, LOAD_KCONTIG)
    TV_CASE(LOAD_MNCONTIG, LOAD_MNCONTIG)
    TV_CASE(LOAD_MNCONTIG, LOAD_KCONTIG)
#undef TV_CASE
    return TV_E_UNSUPPORTED;
}

} // namespace tvk
