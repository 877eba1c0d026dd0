// Products of at most 128 x 128 outputs and K <= 128 (fp32, bf16, fp16, int8; any strides, any sizes).
//
// What bounds them is the launch and one trip to memory; the tiles of the large kernels add a pipeline's
// start and, for rows that are not whole 16-byte chunks, a load per element that waits for the one
// before.  Here a workgroup computes 16 x 16 outputs, one per thread: all of its operands' elements are
// loaded at once (at most 16 loads per thread, all in flight together), widened into LDS, multiplied on
// the vector units and stored.  16-bit sums run in fused fp32 chains of 32 k, added in order, fp32 ones in
// fp64 (as cheap here, and at few k the matrix cores' four products per rounding are not to be lost);
// int8 is exact.
// K of at most 32 or 64 has its own instantiation: with 128 k laid out whatever K, threads along k loaded 16
// elements of which K = 16 used two, and the workgroup held 37 KB of LDS (fp32): fp32 [198][10,32]@Wt[32,48] 5.6 us, bf16 [102]
// [16,16]@Wt[16,80] 4.9, where the kernels of 128 rows took 3.5.
// Measured on 500 random calls of 1 to 128 rows, columns and k (in a captured graph; an empty launch takes about 2.3 us),
// the geometric mean of this kernel's time over that of the kernels that serve the call without it:
//   K            1-32   33-64   65-128
//   unaligned    0.33   0.41    0.40    (fp32 0.36, 0.50, 0.36; 16-bit 0.37, 0.42, 0.46; int8 0.25, 0.28, 0.33)
//   aligned      0.71   0.87    1.20    (fp32 0.72, 0.86, 1.11; 16-bit 0.75, 1.00, 1.39; int8 0.63, 0.81, 1.12)
#include "tv_kernels.h"

namespace tvk {
namespace tiny {

constexpr int kTile = 16, kMaxK = 128, kPitchB = kTile + 4;
constexpr int kMaxDim = 128;

// KM: the most k (32, 64 or 128): what K does not need is neither loaded nor laid out.
template <typename T, typename Acc, int KM>
__global__ __launch_bounds__(256) void gemm_tiny_kernel(GemmDesc d, int tiles_m, int tiles_n) {
    typedef Acc Acc4 __attribute__((ext_vector_type(4)));
    constexpr int NE = KM / 16; // elements per thread and operand
    __shared__ __attribute__((aligned(32))) Acc sa[kTile][KM + 4]; // zero past K and past the rows
    __shared__ __attribute__((aligned(32))) Acc sb[KM][kPitchB];
    const int tid = threadIdx.x;
    const int b = blockIdx.x / (tiles_m * tiles_n), t = blockIdx.x - b * tiles_m * tiles_n;
    const int m0 = t / tiles_n * kTile, n0 = t % tiles_n * kTile;
    const T* A = static_cast<const T*>(d.A) + (int64_t)b * d.sa_b + (int64_t)m0 * d.sa_m;
    const T* B = static_cast<const T*>(d.B) + (int64_t)b * d.sb_b + (int64_t)n0 * d.sb_n;
    // Element e of a thread: consecutive threads along k where k is contiguous, along the rows otherwise.
    const bool ka = d.sa_k == 1, kb = d.sb_k == 1;
    auto k_of = [&](bool kfast, int e) { return kfast ? tid & (KM - 1) : (tid >> 4) + 16 * e; };
    auto r_of = [&](bool kfast, int e) { return kfast ? tid / KM + 256 / KM * e : tid & (kTile - 1); };
    T ra[NE], rb[NE];
#pragma unroll
    for (int e = 0; e < NE; ++e) {
        const int k = k_of(ka, e), r = r_of(ka, e);
        ra[e] = m0 + r < d.M && k < d.K ? A[r * d.sa_m + k * d.sa_k] : T(0);
    }
#pragma unroll
    for (int e = 0; e < NE; ++e) {
        const int k = k_of(kb, e), r = r_of(kb, e);
        rb[e] = n0 + r < d.N && k < d.K ? B[r * d.sb_n + k * d.sb_k] : T(0);
    }
#pragma unroll
    for (int e = 0; e < NE; ++e) {
        sa[r_of(ka, e)][k_of(ka, e)] = static_cast<Acc>(ra[e]);
        sb[k_of(kb, e)][r_of(kb, e)] = static_cast<Acc>(rb[e]);
    }
    __syncthreads();
    const int r = tid >> 4, c = tid & 15;
    Acc v = 0;
    for (int k0 = 0; k0 < d.K; k0 += 32) {
        Acc s = 0;
#pragma unroll
        for (int k = k0; k < k0 + 32; k += 4) {
            const Acc4 x = *reinterpret_cast<const Acc4*>(&sa[r][k]);
            const Acc4 y = {sb[k][c], sb[k + 1][c], sb[k + 2][c], sb[k + 3][c]};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if constexpr (__is_same(Acc, float)) s = __builtin_fmaf(x[q], y[q], s);
                else if constexpr (__is_same(Acc, double)) s = __builtin_fma(x[q], y[q], s);
                else s += x[q] * y[q];
            }
        }
        v = k0 == 0 ? s : v + s;
    }
    const int m = m0 + r, n = n0 + c;
    if (m >= d.M || n >= d.N) return;
    const int64_t i = (int64_t)b * d.sc_b + m * d.sc_m + n * d.sc_n;
    if constexpr (__is_same(Acc, int)) {
        if (d.dtype_c == TV_INT8) static_cast<int8_t*>(d.C)[i] = static_cast<int8_t>(v);
        else static_cast<int32_t*>(d.C)[i] = v;
    } else {
        float f = (float)v;
        if (has_epilogue(d)) f = epilogue_value(f, d, b, m, n);
        if (d.dtype_c == TV_BFLOAT16) static_cast<__bf16*>(d.C)[i] = static_cast<__bf16>(f);
        else if (d.dtype_c == TV_FLOAT16) static_cast<_Float16*>(d.C)[i] = static_cast<_Float16>(f);
        else static_cast<float*>(d.C)[i] = f;
    }
}

} // namespace tiny

// TV_E_UNSUPPORTED above its sizes, or for more workgroups than run at once (the batched kernels serve
// many small products).
int launch_gemm_tiny(const GemmDesc& d, hipStream_t stream) {
    if ((d.bias != nullptr || d.act != TV_ACT_NONE) && d.sc_n != 1) return TV_E_UNSUPPORTED; // as the other kernels
    if (d.M > tiny::kMaxDim || d.N > tiny::kMaxDim || d.K > tiny::kMaxK || d.K < 1) return TV_E_UNSUPPORTED;
    // Operands in whole 16-byte rows have the direct-load kernels, which are faster above 64 k (16-bit: as fast
    // from 33 k; the table above).
    const int es = (int)dtype_size(d.dtype_a);
    if (d.K > (es == 2 ? 32 : 64) && pick_mode(d.A, d.M, d.K, d.sa_m, d.sa_k, d.sa_b, d.batch, es, 256, false) != LOAD_GENERIC &&
        pick_mode(d.B, d.N, d.K, d.sb_n, d.sb_k, d.sb_b, d.batch, es, 256, false) != LOAD_GENERIC)
        return TV_E_UNSUPPORTED;
    const int tm = (d.M + 15) / 16, tn = (d.N + 15) / 16;
    const int64_t blocks = (int64_t)tm * tn * d.batch;
    if (blocks > 4 * (int64_t)device_cus()) return TV_E_UNSUPPORTED;
#define TV_TINY_K(T_, ACC_, KM_) \
    hipLaunchKernelGGL((tiny::gemm_tiny_kernel<T_, ACC_, KM_>), dim3((unsigned)blocks), dim3(256), 0, stream, d, tm, tn)
#define TV_TINY(T_, ACC_)                          \
    if (d.K <= 32) TV_TINY_K(T_, ACC_, 32);        \
    else if (d.K <= 64) TV_TINY_K(T_, ACC_, 64);   \
    else TV_TINY_K(T_, ACC_, 128);                 \
    return hipGetLastError();
    switch (d.dtype_a) {
        case TV_FLOAT32: TV_TINY(float, double)
        case TV_BFLOAT16: TV_TINY(__bf16, float)
        case TV_FLOAT16: TV_TINY(_Float16, float)
        case TV_INT8: TV_TINY(int8_t, int)
        default: return TV_E_UNSUPPORTED;
    }
#undef TV_TINY
#undef TV_TINY_K
}

} // namespace tvk
