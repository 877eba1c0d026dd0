// SIMT path for the dtype pairs the matrix cores do not serve (int16/int32/int64 and mixed pairs;
// fp64 with fp64 runs on gemm_f64.hip).  It restates the reference CPU backend's arithmetic exactly,
// reading operands through their strides, in 64 x 64 tiles or with a thread per output (each_output):
//   * fp16/bf16 inputs are widened to fp32 first (src/backend/cpu/mul.cpp:110-111);
//   * the result type is compute_type of the widened types (mul.cpp:112,
//     include/core/type_traits.h:270-287);
//   * batch*M*N < 2^20 selects mul_kernel_basic (mul.cpp:87-96): the sum runs in
//     decltype(T + R) (mul.cpp:13-18) and is converted to the result type once (mul.cpp:21);
//   * otherwise mul_kernel_tiled<.., 64> (mul.cpp:27-85): each 64-wide k-chunk is summed in A's
//     type T with B's values converted to T (mul.cpp:64-71), and chunk sums are converted to the
//     result type and added into it (mul.cpp:74-78).
// Integer arithmetic wraps (two's complement), as the reference's does on its targets; float to
// integer conversion of out-of-range values yields the x86 "integer indefinite" value.
#include "tv_kernels.h"

namespace tvk {
namespace simt {

template <typename X> struct Promote { using type = X; };
template <> struct Promote<int8_t> { using type = int; };
template <> struct Promote<int16_t> { using type = int; };
template <typename A, typename B>
using Common = decltype(typename Promote<A>::type{} + typename Promote<B>::type{});

template <bool C, typename A, typename B> struct Pick { using type = A; };
template <typename A, typename B> struct Pick<false, A, B> { using type = B; };

template <typename X> struct Unsigned;
template <> struct Unsigned<int8_t> { using type = uint8_t; };
template <> struct Unsigned<int16_t> { using type = uint16_t; };
template <> struct Unsigned<int> { using type = unsigned; };
template <> struct Unsigned<long> { using type = unsigned long; };
template <> struct Unsigned<long long> { using type = unsigned long long; };

template <typename X> __device__ constexpr bool is_int() { return !__is_same(X, float) && !__is_same(X, double); }

// static_cast<To>(from) with the reference targets' behaviour for every case.
template <typename To, typename From> __device__ inline To cvt(From v) {
    if constexpr (is_int<To>() && !is_int<From>()) {
        const double x = (double)v;
        if constexpr (sizeof(To) == 8) {
            if (!(x > -9223372036854775808.0 - 1.0 && x < 9223372036854775808.0)) return (To)(int64_t)(-9223372036854775807LL - 1);
            return (To)(int64_t)x;
        } else {
            if (!(x > -2147483649.0 && x < 2147483648.0)) return (To)(int32_t)(-2147483647 - 1);
            return (To)(int32_t)x;
        }
    } else {
        return static_cast<To>(v);
    }
}

template <typename X> __device__ inline X add(X a, X b) {
    if constexpr (is_int<X>()) {
        using U = typename Unsigned<X>::type;
        return (X)(U)((U)a + (U)b);
    } else {
        return a + b;
    }
}
template <typename X> __device__ inline X mul(X a, X b) {
    if constexpr (is_int<X>()) {
        using U = typename Unsigned<X>::type;
        return (X)(U)((U)a * (U)b);
    } else {
        return a * b;
    }
}

// acc (type Acc) += x * y with the C++ promotions of `Acc += P * P`.
template <typename Acc, typename P> __device__ inline Acc mac(Acc acc, P x, P y) {
    using Prod = typename Promote<P>::type;
    const Prod p = mul<Prod>((Prod)x, (Prod)y);
    using Sum = Common<Acc, Prod>;
    return cvt<Acc>(add<Sum>((Sum)acc, (Sum)p));
}

// Storage of an operand whose widened type is T: T itself, except that float also stands for fp16
// and bf16 storage.  Raw<T> holds one element as loaded (16-bit elements zero-extended), so that a
// batch of loads stays in flight until its elements are converted.
template <typename T> struct RawOf { using type = T; };
template <> struct RawOf<float> { using type = unsigned; };
template <typename T> using Raw = typename RawOf<T>::type;

// dst[e] = the element of storage type dt at ptr(e); one uniform branch for the whole batch.
template <typename T, int N, class Ptr> __device__ inline void load_raw(int dt, Raw<T> (&dst)[N], const Ptr& ptr) {
    if constexpr (__is_same(T, float)) {
        if (dt == TV_FLOAT32) {
#pragma unroll
            for (int e = 0; e < N; ++e) dst[e] = *reinterpret_cast<const unsigned*>(ptr(e));
        } else {
#pragma unroll
            for (int e = 0; e < N; ++e) dst[e] = *reinterpret_cast<const unsigned short*>(ptr(e));
        }
    } else {
#pragma unroll
        for (int e = 0; e < N; ++e) dst[e] = *reinterpret_cast<const T*>(ptr(e));
    }
}
// put(e, widened element e) for a loaded batch.
template <typename T, int N, class Put> __device__ inline void widen_raw(int dt, const Raw<T> (&src)[N], const Put& put) {
    if constexpr (__is_same(T, float)) {
        if (dt == TV_FLOAT32) {
#pragma unroll
            for (int e = 0; e < N; ++e) put(e, __builtin_bit_cast(float, src[e]));
        } else if (dt == TV_BFLOAT16) {
#pragma unroll
            for (int e = 0; e < N; ++e) put(e, __builtin_bit_cast(float, src[e] << 16));
        } else {
#pragma unroll
            for (int e = 0; e < N; ++e) put(e, (float)__builtin_bit_cast(_Float16, (unsigned short)src[e]));
        }
    } else {
#pragma unroll
        for (int e = 0; e < N; ++e) put(e, src[e]);
    }
}

template <typename S> __device__ inline void store_as(void* p, int dt, int64_t idx, S v) {
    switch (dt) {
        case TV_INT8: static_cast<int8_t*>(p)[idx] = cvt<int8_t>(v); break;
        case TV_INT16: static_cast<int16_t*>(p)[idx] = cvt<int16_t>(v); break;
        case TV_INT32: static_cast<int32_t*>(p)[idx] = cvt<int32_t>(v); break;
        case TV_INT64: static_cast<long*>(p)[idx] = cvt<long>(v); break;
        case TV_FLOAT32: static_cast<float*>(p)[idx] = cvt<float>(v); break;
        default: static_cast<double*>(p)[idx] = cvt<double>(v); break;
    }
}

// Result type of the widened pair (T, R): compute_type (include/core/type_traits.h:270-287).
template <typename T, typename R> constexpr auto result_value() {
    if constexpr (__is_same(T, R)) return T{};
    else if constexpr (is_int<T>() && is_int<R>()) {
        if constexpr (sizeof(T) > sizeof(R)) return T{};
        else return R{};
    } else if constexpr (__is_same(T, double) || __is_same(R, double) || __is_same(T, long) || __is_same(R, long)) return double{};
    else return float{};
}

// One workgroup computes 64 x 64 outputs, a thread 4 x 4 of them, summing k in order as the CPU
// kernels do: every output's sum is the one thread's of a thread per output, bit for bit.  What
// bounds the pairs is the VALU (fp32: one FMA per output and k; 32-bit integers: the quarter-rate
// multiply), if operands are reused: with a thread per output, each multiply-add waited for two
// loads from memory (0.3 us per k however small the call, 1.3 ms for 1000^3 in fp64).  Here 32 k of
// both operands are converted once into LDS (two stages; the next 32 k are loaded into registers
// while the current ones are multiplied, one barrier per 32 k), and a thread's 16 multiply-adds per
// k read two 4-element vectors.  Against a thread per output, same box (us): fp32 x bf16
// [1024,600]@[600,1024] 710 -> 47 (26 TFLOP/s), fp32 x fp16 [1000,600]@Wt[1000,600] 2390 -> 49,
// int32 [1000,600]@[600,1000] 637 -> 55, int16 630 -> 53, fp32 x bf16 x[1,4096]@W[4096,4096]
// 1753 -> 279, fp32 x fp16 [37,64]@[64,448] 21.4 -> 9.2.
// X: the type the products run in: decltype(T + R), or T in the chunked sums (TILED).
constexpr int kTile = 64, kBk = 32, kPitch = kTile + 4; // k rows of 64 elements, padded
template <typename T, typename R, typename S, bool TILED>
__global__ __launch_bounds__(256) void gemm_simt_kernel(GemmDesc d, int64_t tiles_m, int64_t tiles_n) {
    using P = Common<T, R>;
    using X = typename Pick<TILED, T, P>::type;
    typedef X X4 __attribute__((ext_vector_type(4)));
    static_assert(64 % kBk == 0, "a chunk is whole k-tiles");
    __shared__ __attribute__((aligned(32))) X sa[2][kBk][kPitch];
    __shared__ __attribute__((aligned(32))) X sb[2][kBk][kPitch];
    constexpr int NE = kTile * kBk / 256; // elements per thread, operand and k-tile
    const int tid = threadIdx.x;
    const int tx = tid & 15, ty = tid >> 4;
    // Consecutive threads along whichever dimension is contiguous: (row, k) of element e.
    const bool ka = d.sa_k == 1, kb = d.sb_k == 1;
    auto row_of = [&](bool kfast, int e) { return kfast ? (tid >> 5) + 8 * e : (tid & 63); };
    auto k_of = [&](bool kfast, int e) { return kfast ? (tid & 31) : (tid >> 6) + 4 * e; };
    const int64_t ntiles = tiles_m * tiles_n * d.batch;
    const int nk = (d.K + kBk - 1) / kBk;
    const int64_t esa = dtype_size(d.dtype_a), esb = dtype_size(d.dtype_b);

    for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const int64_t b = t / (tiles_m * tiles_n), r = t - b * tiles_m * tiles_n;
        const int64_t m0 = r / tiles_n * kTile, n0 = r % tiles_n * kTile;
        Raw<T> ra[NE];
        Raw<R> rb[NE];
        // Element pointers at k-tile 0.  Rows past the matrix re-read its last row (their outputs are
        // not stored); elements past K re-read k = 0 of the row and are not multiplied.
        const char* pa[NE];
        const char* pb[NE];
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            pa[e] = static_cast<const char*>(d.A) + (b * d.sa_b + min(m0 + row_of(ka, e), (int64_t)d.M - 1) * d.sa_m) * esa;
            pb[e] = static_cast<const char*>(d.B) + (b * d.sb_b + min(n0 + row_of(kb, e), (int64_t)d.N - 1) * d.sb_n) * esb;
        }
        auto load = [&](int kt) {
            load_raw<T>(d.dtype_a, ra, [&](int e) {
                const int k = kt * kBk + k_of(ka, e);
                return pa[e] + (k < d.K ? k : 0) * d.sa_k * esa;
            });
            load_raw<R>(d.dtype_b, rb, [&](int e) {
                const int k = kt * kBk + k_of(kb, e);
                return pb[e] + (k < d.K ? k : 0) * d.sb_k * esb;
            });
        };
        auto store = [&](int st) {
            widen_raw<T>(d.dtype_a, ra, [&](int e, T v) { sa[st][k_of(ka, e)][row_of(ka, e)] = cvt<X>(v); });
            widen_raw<R>(d.dtype_b, rb, [&](int e, R v) { sb[st][k_of(kb, e)][row_of(kb, e)] = cvt<X>(v); });
        };
        X sum[4][4];
        S res[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) sum[i][j] = 0, res[i][j] = 0;
        auto read = [&](int st, int k, X4& x, X4& y) {
            x = *reinterpret_cast<const X4*>(&sa[st][k][4 * ty]);
            y = *reinterpret_cast<const X4*>(&sb[st][k][4 * tx]);
        };
        auto macs = [&](const X4& x, const X4& y) {
            const X xs[4] = {x[0], x[1], x[2], x[3]}, ys[4] = {y[0], y[1], y[2], y[3]};
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) sum[i][j] = mac<X, X>(sum[i][j], xs[i], ys[j]);
        };
        if (nk > 0) {
            load(0);
            store(0);
            load(1);
        }
        __syncthreads();
        for (int kt = 0; kt < nk; ++kt) {
            const int st = kt & 1;
            store(st ^ 1); // read last in step kt - 1, before its barrier
            load(kt + 2);
            const int kn = min(kBk, d.K - kt * kBk);
            if (kn == kBk) {
                // The next G k's operands are read while the current G are multiplied: left to
                // itself the compiler waited for each k's reads right after issuing them.
                constexpr int G = sizeof(X) == 8 ? 2 : 4;
                X4 x[2][G], y[2][G];
#pragma unroll
                for (int u = 0; u < G; ++u) read(st, u, x[0][u], y[0][u]);
#pragma unroll
                for (int g = 0; g < kBk / G; ++g) {
                    if (g + 1 < kBk / G) {
#pragma unroll
                        for (int u = 0; u < G; ++u) read(st, (g + 1) * G + u, x[(g + 1) & 1][u], y[(g + 1) & 1][u]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int u = 0; u < G; ++u) macs(x[g & 1][u], y[g & 1][u]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
                for (int k = 0; k < kn; ++k) {
                    X4 x, y;
                    read(st, k, x, y);
                    macs(x, y);
                }
            }
            if constexpr (TILED) {
                if ((kt + 1) % (64 / kBk) == 0 || kt + 1 == nk) { // the end of a 64-wide chunk
                    const bool first = (kt + 1) * kBk <= 64;
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const S c = cvt<S>(sum[i][j]);
                            res[i][j] = first ? c : cvt<S>(add<Common<S, S>>((Common<S, S>)res[i][j], (Common<S, S>)c));
                            sum[i][j] = 0;
                        }
                }
            }
            __syncthreads();
        }
        S* C = static_cast<S*>(d.C) + b * d.sc_b;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int64_t m = m0 + 4 * ty + i, n = n0 + 4 * tx + j;
                if (m < d.M && n < d.N) C[m * d.sc_m + n * d.sc_n] = TILED ? res[i][j] : cvt<S>(sum[i][j]);
            }
    }
}

// One thread per output, for batches of small matrices and thin ones, whose tiles would be mostly empty.  What
// bounds it is the latency of its loads (16 of them, 8 k, are in flight per thread: 0.05 us per k where all
// outputs run at once, 0.2 with one pair of loads waited for at a time), then the lines that a wave's loads
// touch.  Sums run in the order of the tiled kernels: the results are theirs bit for bit.
template <typename T, typename R, typename S, bool TILED, typename IDX>
__global__ __launch_bounds__(256) void gemm_each_kernel(GemmDesc d, IDX total) {
    using P = Common<T, R>;
    using X = typename Pick<TILED, T, P>::type;
    const IDX N = (IDX)d.N, M = (IDX)d.M, stride = (IDX)gridDim.x * 256;
    const int64_t esa = dtype_size(d.dtype_a), esb = dtype_size(d.dtype_b), ska = d.sa_k * esa, skb = d.sb_k * esb;
    for (IDX o = (IDX)blockIdx.x * 256 + threadIdx.x; o < total; o += stride) {
        const IDX row = o / N, n = o - row * N, b = row / M, m = row - b * M;
        const char* pa = static_cast<const char*>(d.A) + ((int64_t)b * d.sa_b + (int64_t)m * d.sa_m) * esa;
        const char* pb = static_cast<const char*>(d.B) + ((int64_t)b * d.sb_b + (int64_t)n * d.sb_n) * esb;
        X sum = 0;
        S res = 0;
        auto products = [&]<int G>(int k) { // G products from k on, their elements loaded at once
            Raw<T> ra[G];
            Raw<R> rb[G];
            X x[G], y[G];
            load_raw<T>(d.dtype_a, ra, [&](int e) { return pa + (int64_t)(k + e) * ska; });
            load_raw<R>(d.dtype_b, rb, [&](int e) { return pb + (int64_t)(k + e) * skb; });
            widen_raw<T>(d.dtype_a, ra, [&](int e, T v) { x[e] = cvt<X>(v); });
            widen_raw<R>(d.dtype_b, rb, [&](int e, R v) { y[e] = cvt<X>(v); });
#pragma unroll
            for (int e = 0; e < G; ++e) sum = mac<X, X>(sum, x[e], y[e]);
        };
        for (int k0 = 0; k0 < d.K; k0 += 64) {
            const int end = k0 + min(d.K - k0, 64);
            int k = k0;
            for (; k + 8 <= end; k += 8) products.template operator()<8>(k);
            if (k + 4 <= end) products.template operator()<4>(k), k += 4;
            if (k + 2 <= end) products.template operator()<2>(k), k += 2;
            if (k < end) products.template operator()<1>(k);
            if constexpr (TILED) {
                const S c = cvt<S>(sum);
                res = k0 == 0 ? c : cvt<S>(add<Common<S, S>>((Common<S, S>)res, (Common<S, S>)c));
                sum = 0;
            }
        }
        static_cast<S*>(d.C)[(int64_t)b * d.sc_b + (int64_t)m * d.sc_m + (int64_t)n * d.sc_n] = TILED ? res : cvt<S>(sum);
    }
}

static int widen(int dt) { return (dt == TV_BFLOAT16 || dt == TV_FLOAT16) ? TV_FLOAT32 : dt; }

// Whether a thread per output is cheaper than a tile per workgroup: every matrix costs at least one whole tile,
// so batches of small matrices and thin ones pay for 64 x 64 outputs that they do not have (fp64
// [100000][4,4]@[4,4] 2,156 us on tiles, 11 here; int32 [10000][8,8]@[8,8] 170, 7; fp64 [1000000,3]@[3,3] 356, 22).
// Both prices, in us, are fitted to 1,800 random calls (1 to 200,000 matrices of 1 to 500,000 rows or columns, K of 1 to
// 4096) timed both ways.  The first is the less certain one (how many lines of A and B the L1 keeps), most where
// latency bounds it, so the tiles are kept unless it is that much less.
static bool each_output(const GemmDesc& d) {
    const double cus = device_cus(), K = d.K, total = (double)d.batch * d.M * d.N;
    auto tiles = [&](int t) { return (double)(((int64_t)d.M + t - 1) / t) * (double)(((int64_t)d.N + t - 1) / t) * d.batch; };
    auto over = [](double tiles, double held) { return tiles > held ? tiles / held : 1.0; };
    // Lanes on consecutive columns of a row-major B share its lines; rows of fewer than a wave's columns take lines
    // of several rows of A, and a B contiguous along k a line per lane, which the L1 seldom keeps until the next k.
    const bool b_lines = d.sb_n != 1 && d.N > 1, lines = b_lines || d.N < 64;
    const double k_us = b_lines ? 0.13 : lines ? 0.089 : 0.058;
    const double mac_us = b_lines || d.N < 16 ? 1.5e-6 : lines ? 1.0e-6 : 0.68e-6;
    const double each = 1.9 + K * (total * mac_us > k_us ? total * mac_us : k_us);
    double tile;
    if (d.dtype_a == TV_FLOAT64 && d.dtype_b == TV_FLOAT64) {
        const int t = f64_tile(d);
        const double n = tiles(t) / cus, steps = 2.0 * ((d.K + 63) / 64);
        tile = t == 64 ? 3.3 + 2.6 * n + steps * (n > 0.8 ? 1.6 * n : 1.3) : 3.3 + 1.6 * n + steps * (n > 0.8 ? 0.57 * n : 0.46);
    } else {
        const bool i64 = d.dtype_a == TV_INT64 || d.dtype_b == TV_INT64;
        const double n = tiles(kTile);
        tile = 5.0 + 2.75 * (i64 ? 1.8 : 1.0) * K / kBk * over(n, 0.96 * cus) + 3.9 * n / cus;
    }
    return (total * mac_us > k_us ? 1.15 : 1.3) * each < tile;
}

template <typename T, typename R, typename S, bool TILED>
static int launch_each(const GemmDesc& d, hipStream_t stream) {
    const int64_t total = (int64_t)d.batch * d.M * d.N, blocks = (total + 255) / 256;
    const unsigned grid = blocks < 65536 ? (unsigned)blocks : 65536u;
    if (total < ((int64_t)1 << 31))
        hipLaunchKernelGGL((gemm_each_kernel<T, R, S, TILED, uint32_t>), dim3(grid), dim3(256), 0, stream, d, (uint32_t)total);
    else
        hipLaunchKernelGGL((gemm_each_kernel<T, R, S, TILED, int64_t>), dim3(grid), dim3(256), 0, stream, d, total);
    return hipGetLastError();
}

template <typename T, typename R>
static int launch_tr(const GemmDesc& d, hipStream_t stream) {
    using S = decltype(result_value<T, R>());
    const bool chunked = (__int128)d.batch * d.M * d.N >= 1024 * 1024; // mul_kernel_tiled
    if (each_output(d)) return chunked ? launch_each<T, R, S, true>(d, stream) : launch_each<T, R, S, false>(d, stream);
    if constexpr (__is_same(T, double) && __is_same(R, double)) {
        return launch_gemm_f64(d, stream);
    } else {
        const int64_t tiles_m = ((int64_t)d.M + kTile - 1) / kTile, tiles_n = ((int64_t)d.N + kTile - 1) / kTile;
        // Up to 2^25 x 2^25 tiles and 2^31 batches: the grid is capped and a workgroup takes every
        // grid-size-th tile; a count past 2^62 could never run.
        const __int128 n = (__int128)tiles_m * tiles_n * d.batch;
        if (n > ((__int128)1 << 62)) return TV_E_SHAPE;
        const unsigned blocks = n < ((int64_t)1 << 20) ? (unsigned)n : 1u << 20;
        if (chunked)
            hipLaunchKernelGGL((gemm_simt_kernel<T, R, S, true>), dim3(blocks), dim3(256), 0, stream, d, tiles_m, tiles_n);
        else
            hipLaunchKernelGGL((gemm_simt_kernel<T, R, S, false>), dim3(blocks), dim3(256), 0, stream, d, tiles_m, tiles_n);
        return hipGetLastError();
    }
}

template <typename T>
static int launch_t(const GemmDesc& d, hipStream_t stream) {
    switch (widen(d.dtype_b)) {
        case TV_INT8:
            if constexpr (!__is_same(T, int8_t)) return launch_tr<T, int8_t>(d, stream);
            else return TV_E_DTYPE; // int8 x int8 runs on the matrix cores
        case TV_INT16: return launch_tr<T, int16_t>(d, stream);
        case TV_INT32: return launch_tr<T, int>(d, stream);
        case TV_INT64: return launch_tr<T, long>(d, stream);
        case TV_FLOAT32: return launch_tr<T, float>(d, stream);
        case TV_FLOAT64: return launch_tr<T, double>(d, stream);
        default: return TV_E_DTYPE;
    }
}

// K = 0: every output is the empty sum, through the fused epilogue when one is given (act(bias)).
__global__ __launch_bounds__(256) void gemm_k0_kernel(GemmDesc d) {
    const int64_t total = (int64_t)d.batch * d.M * d.N;
    for (int64_t o = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; o < total; o += (int64_t)gridDim.x * blockDim.x) {
        const int64_t n = o % d.N;
        const int64_t m = (o / d.N) % d.M;
        const int64_t b = o / ((int64_t)d.N * d.M);
        const float v = has_epilogue(d) ? epilogue_value(0.0f, d, b, m, n) : 0.0f;
        const int64_t i = b * d.sc_b + m * d.sc_m + n * d.sc_n;
        switch (d.dtype_c) {
            case TV_BFLOAT16: static_cast<__bf16*>(d.C)[i] = static_cast<__bf16>(v); break;
            case TV_FLOAT16: static_cast<_Float16*>(d.C)[i] = static_cast<_Float16>(v); break;
            case TV_FLOAT32: static_cast<float*>(d.C)[i] = v; break;
            default: store_as<int>(d.C, d.dtype_c, i, 0); break;
        }
    }
}

} // namespace simt

int launch_gemm_k0(const GemmDesc& d, hipStream_t stream) {
    const int64_t total = (int64_t)d.batch * d.M * d.N;
    if (total == 0) return 0;
    int64_t blocks = (total + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(simt::gemm_k0_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, d);
    return hipGetLastError();
}

int launch_gemm_simt(const GemmDesc& d, hipStream_t stream) {
    if ((int64_t)d.batch * d.M * d.N == 0) return 0;
    switch (simt::widen(d.dtype_a)) {
        case TV_INT8: return simt::launch_t<int8_t>(d, stream);
        case TV_INT16: return simt::launch_t<int16_t>(d, stream);
        case TV_INT32: return simt::launch_t<int>(d, stream);
        case TV_INT64: return simt::launch_t<long>(d, stream);
        case TV_FLOAT32: return simt::launch_t<float>(d, stream);
        case TV_FLOAT64: return simt::launch_t<double>(d, stream);
        default: return TV_E_DTYPE;
    }
}

} // namespace tvk
