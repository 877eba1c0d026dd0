// fp64 matmul on the fp64 matrix cores (v_mfma_f64_16x16x4_f64), any strides.
//
// Replaces MulImpl's loops for double x double (reference src/backend/cpu/mul.cpp:7-85) and sums in
// their order: k in sequence, and from batch*M*N = 2^20 (mul_kernel_tiled, mul.cpp:64-78,87-96) each
// 64-wide k-chunk by itself, then added to the output.
//
// What bounds it: the fp64 matrix rate (as high as the vector one, 64 FMAs per CU and cycle), if the
// operands reach it.  A vector kernel would be LDS-bound: a 4 x 4 block per thread reads 64 bytes for
// 16 FMAs, twice what LDS delivers in the FMAs' time.  The matrix instruction needs one A and one B
// value per lane for 16 FMAs, and a wave's 32 x 16 block (2 x 1 instructions) uses each of B's twice.
//  * A workgroup computes TILE x TILE outputs, TILE = 64 (8 waves of 32 x 16, two per SIMD) or 32 (4
//    waves of 16 x 16).
//  * 32 k of each operand per step, in LDS rows of one output row or column each.  Two LDS stages and
//    two steps ahead in registers, one barrier per step.
//  * A lane reads two k at once (16 bytes), k = 8s + lane/16 and 8s + 4 + lane/16, which rows of LDS
//    hold side by side: the halves go to two instructions, each summing 4 consecutive k.
//  * Tiles are walked in groups of 4 tile-rows, consecutive ones on one XCD, which then streams 12
//    panels per 32 tiles through its L2 instead of 18.
// Measured against the thread-per-output kernel before it, same box: [1000]^3 1,302 -> 46 us (44
// TFLOP/s; the library's large product reaches 72), the same with B a transposed view 4,042 -> 46,
// [1280,600]@[600,1280] 1,275 -> 60, [320,600]@[600,320] 249 -> 13, [64]^3 21.9 -> 4.5.
#include "gemm_mfma_impl.h"

namespace tvk {
namespace f64 {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
constexpr int kBk = 32;        // k per step

constexpr int kGroupM = 4;

template <int TILE, bool CHUNKS>
__global__ __launch_bounds__(TILE == 64 ? 512 : 256, 2) void gemm_f64_kernel(GemmDesc d, int tiles_m, int tiles_n, int ntiles) {
    constexpr int THREADS = TILE == 64 ? 512 : 256;
    constexpr int WN_WAVES = THREADS / 128;     // waves: 2 x WN_WAVES
    constexpr int WM = TILE / 2, WN = TILE / WN_WAVES, FM = WM / 16, FN = WN / 16;
    constexpr int NE = TILE * kBk / THREADS;    // elements per thread, operand and step
    __shared__ __attribute__((aligned(16))) double sa[2][TILE][kBk];
    __shared__ __attribute__((aligned(16))) double sb[2][TILE][kBk];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = (wave / WN_WAVES) * WM, wn = (wave % WN_WAVES) * WN;
    const int fr = lane & 15, kg = lane >> 4;
    // Consecutive threads along whichever dimension is contiguous: (row, k) of element e.
    const bool ka = d.sa_k == 1, kb = d.sb_k == 1;
    auto row_of = [&](bool kfast, int e) { return kfast ? (tid >> 5) + THREADS / 32 * e : tid % TILE; };
    auto k_of = [&](bool kfast, int e) { return kfast ? (tid & 31) : tid / TILE + THREADS / TILE * e; };
    static_assert(NE == kBk / 8, "one element per 8 k of a step");
    // Place of k in LDS row r: k and k + 4 of a group of 8 side by side, and the 16-byte pair p of the
    // row at p ^ (r % 16), so neither the row-wise nor the column-wise accesses conflict.
    auto pos = [](int k, int r) { return (((((k >> 3) << 2) | (k & 3)) ^ (r & 15)) << 1) | ((k >> 2) & 1); };

    int id = blockIdx.x;
    if ((ntiles & 7) == 0) id = (id & 7) * (ntiles >> 3) + (id >> 3);
    int b, tm, tn;
    mfma_tile_of(id, tiles_m, tiles_n, kGroupM, b, tm, tn);
    const int64_t m0 = (int64_t)tm * TILE, n0 = (int64_t)tn * TILE;
    const double* A = static_cast<const double*>(d.A) + (int64_t)b * d.sa_b + m0 * d.sa_m;
    const double* B = static_cast<const double*>(d.B) + (int64_t)b * d.sb_b + n0 * d.sb_n;
    const int nk = (d.K + kBk - 1) / kBk;

    // Pointers of the element each thread loads next (element e: row row_of(e), k k_of(e) of the step),
    // advanced by a step's k after each load.  Rows past the matrix re-read its last row (their outputs
    // are not stored); elements past K re-read k = 0 of the row and are zeroed on their way into LDS.
    // Every step issues the same loads without a branch, so the waits count them exactly.
    const double* pa[NE];
    const double* pb[NE];
    const double* ra0[NE];
    const double* rb0[NE];
#pragma unroll
    for (int e = 0; e < NE; ++e) {
        ra0[e] = A + min((int64_t)row_of(ka, e), d.M - 1 - m0) * d.sa_m;
        rb0[e] = B + min((int64_t)row_of(kb, e), d.N - 1 - n0) * d.sb_n;
        pa[e] = ra0[e] + k_of(ka, e) * d.sa_k;
        pb[e] = rb0[e] + k_of(kb, e) * d.sb_k;
    }
    const int64_t inc_a = kBk * d.sa_k, inc_b = kBk * d.sb_k;
    double ra[2][NE], rb[2][NE];
    auto load = [&](int set, int e, int kt) {
        ra[set][e] = *(kt * kBk + k_of(ka, e) < d.K ? pa[e] : ra0[e]);
        rb[set][e] = *(kt * kBk + k_of(kb, e) < d.K ? pb[e] : rb0[e]);
        pa[e] += inc_a;
        pb[e] += inc_b;
    };
    auto store = [&](int st, int set, int e, int kt) {
        const int k = k_of(ka, e), kk = k_of(kb, e), i = row_of(ka, e), j = row_of(kb, e);
        sa[st][i][pos(k, i)] = kt * kBk + k < d.K ? ra[set][e] : 0.0;
        sb[st][j][pos(kk, j)] = kt * kBk + kk < d.K ? rb[set][e] : 0.0;
    };
    f64x4 acc[FM][FN], sum[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = f64x4{0, 0, 0, 0}, sum[i][j] = f64x4{0, 0, 0, 0};

    // Step kt multiplies LDS stage kt % 2, stores step kt + 1 (registers, set (kt + 1) % 2) into the
    // other stage, read last in step kt - 1, before its barrier, and loads step kt + 3 into that set.
    // The stores and loads go out a share per 8 k, between the MFMAs (with all of them before the
    // MFMAs, both waves of a SIMD did their address arithmetic at the same time, as long as the
    // MFMAs take), and the next 8 k's fragments are read while the current ones are multiplied.
    auto step = [&](int kt, int st) {
        f64x2 fa[2][FM], fb[2][FN];
        auto read = [&](int s) {
#pragma unroll
            for (int i = 0; i < FM; ++i) fa[s & 1][i] = *reinterpret_cast<const f64x2*>(&sa[st][wm + 16 * i + fr][pos(8 * s + kg, fr)]);
#pragma unroll
            for (int j = 0; j < FN; ++j) fb[s & 1][j] = *reinterpret_cast<const f64x2*>(&sb[st][wn + 16 * j + fr][pos(8 * s + kg, fr)]);
        };
        read(0);
#pragma unroll
        for (int s = 0; s < kBk / 8; ++s) {
            if (s + 1 < kBk / 8) read(s + 1);
            store(st ^ 1, st ^ 1, s, kt + 1);
            load(st ^ 1, s, kt + 3);
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[s & 1][i][h], fb[s & 1][j][h], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (CHUNKS)
            if ((kt + 1) % (64 / kBk) == 0) { // the end of a 64-wide chunk
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j) {
                        sum[i][j] += acc[i][j];
                        acc[i][j] = f64x4{0, 0, 0, 0};
                    }
            }
        __syncthreads();
    };
    if (nk > 0) {
#pragma unroll
        for (int e = 0; e < NE; ++e) load(0, e, 0);
#pragma unroll
        for (int e = 0; e < NE; ++e) load(1, e, 1);
#pragma unroll
        for (int e = 0; e < NE; ++e) store(0, 0, e, 0);
#pragma unroll
        for (int e = 0; e < NE; ++e) load(0, e, 2);
        __syncthreads();
        for (int kt = 0; kt < nk; kt += 2) { // a step past K multiplies zeros
            step(kt, 0);
            step(kt + 1, 1);
        }
    }
    // Element r of a lane's block (i, j) is row 16i + lane/16 + 4r, column 16j + lane%16 of the wave's block.
    double* C = static_cast<double*>(d.C) + (int64_t)b * d.sc_b;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t m = m0 + wm + 16 * i + kg + 4 * r;
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const int64_t n = n0 + wn + 16 * j + fr;
                if (m < d.M && n < d.N) C[m * d.sc_m + n * d.sc_n] = CHUNKS ? sum[i][j][r] : acc[i][j][r];
            }
        }
}

} // namespace f64

static __int128 f64_tiles(const GemmDesc& d, int t) {
    return (__int128)(((int64_t)d.M + t - 1) / t) * (((int64_t)d.N + t - 1) / t) * d.batch;
}

// 64 x 64 tiles when they give at least three quarters of the CUs one; 32 x 32 below that, where
// four times the workgroups each do a quarter of the matrix work per load latency, and where the small
// tiles leave a quarter of the large ones' outputs out (us, 32 x 32 / 64 x 64: [3000][32,64]@[64,32] 33 / 73,
// [400][96,64]@[64,96] 37 / 45, [3000][64,64]@[64,16] 57 / 75; but [3000][40,64]@[64,40] 107 / 75).
int f64_tile(const GemmDesc& d) {
    const __int128 large = f64_tiles(d, 64);
    return large * 4 >= device_cus() * 3 && f64_tiles(d, 32) > 3 * large ? 64 : 32;
}

// chunks: the sum's order, by the whole call's outputs.
static int launch_tiles(const GemmDesc& d, int t, bool chunks, hipStream_t stream) {
    const __int128 n = f64_tiles(d, t);
    const int threads = t == 64 ? 512 : 256;
    if (n * threads > 0xFFFFFFFFll) { // more than one grid holds (2^32 threads): half of the batch or of the rows at a time
        GemmDesc lo = d, hi = d;
        if (d.batch > 1) {
            lo.batch = d.batch / 2;
            hi.batch = d.batch - lo.batch;
            hi.A = static_cast<const double*>(d.A) + lo.batch * d.sa_b;
            hi.B = static_cast<const double*>(d.B) + lo.batch * d.sb_b;
            hi.C = static_cast<double*>(d.C) + lo.batch * d.sc_b;
        } else if (d.M > t) {
            lo.M = (d.M / 2 + t - 1) / t * t;
            hi.M = d.M - lo.M;
            hi.A = static_cast<const double*>(d.A) + lo.M * d.sa_m;
            hi.C = static_cast<double*>(d.C) + lo.M * d.sc_m;
        } else {
            lo.N = (d.N / 2 + t - 1) / t * t;
            hi.N = d.N - lo.N;
            hi.B = static_cast<const double*>(d.B) + lo.N * d.sb_n;
            hi.C = static_cast<double*>(d.C) + lo.N * d.sc_n;
        }
        const int rc = launch_tiles(lo, t, chunks, stream);
        return rc ? rc : launch_tiles(hi, t, chunks, stream);
    }
    const int tm = (int)(((int64_t)d.M + t - 1) / t), tn = (int)(((int64_t)d.N + t - 1) / t);
#define TV_F64(T_, C_)                                                                                                     \
    if (t == T_ && chunks == C_)                                                                                           \
        hipLaunchKernelGGL((f64::gemm_f64_kernel<T_, C_>), dim3((unsigned)n), dim3(T_ == 64 ? 512 : 256), 0, stream, d, tm, \
                           tn, (int)n);
    TV_F64(64, true)
    TV_F64(64, false)
    TV_F64(32, true)
    TV_F64(32, false)
#undef TV_F64
    return hipGetLastError();
}

int launch_gemm_f64(const GemmDesc& d, hipStream_t stream) {
    return launch_tiles(d, f64_tile(d), (__int128)d.batch * d.M * d.N >= 1024 * 1024, stream);
}

} // namespace tvk
