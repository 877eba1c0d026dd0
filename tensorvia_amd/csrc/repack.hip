// Strided view -> contiguous copy (TensorImpl::clone_as_contiguous of the HIP backend, and the
// materialising ops::Transpose).  Restates RepackImpl<Device::CUDA> (reference
// src/backend/cuda/repack.cu:5-54) without its per-call device allocations: shape and strides travel
// in the kernel arguments.  Three kernels, by the view's layout:
//  * rows: the innermost dimension is contiguous in the source and rows are 16-byte aligned; each
//    thread moves 16 bytes, so reads and writes are whole 16-byte accesses;
//  * transpose: the last two dimensions are swapped (source stride 1 on the next-to-last dimension,
//    as K.permute(0, 2, 1)); 64 x 64 element tiles go through LDS, so reads run along the source's
//    contiguous dimension and writes along the destination's (16-bit elements in 4-byte pairs when
//    the view allows);
//  * element: anything else, one element per thread, consecutive threads writing consecutive
//    destination elements.
#include "tv_kernels.h"

namespace tvk {

struct RepackDesc {
    int64_t shape[TV_MAX_DIMS];
    int64_t strides[TV_MAX_DIMS];
    int ndim;
    int64_t numel;
    const void* src;
    void* dst;
};

// Source element offset of the first element of "outer" index o over dimensions [0, nd).
__device__ inline int64_t outer_offset(const RepackDesc& r, int nd, int64_t o) {
    int64_t off = 0;
    for (int d = nd - 1; d >= 0; --d) {
        const int64_t c = o % r.shape[d];
        o /= r.shape[d];
        off += c * r.strides[d];
    }
    return off;
}

template <typename E>
__global__ __launch_bounds__(256) void repack_kernel(RepackDesc r) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < r.numel; i += stride)
        static_cast<E*>(r.dst)[i] = static_cast<const E*>(r.src)[outer_offset(r, r.ndim, i)];
}

// Rows of CPR 16-byte chunks: chunk c of destination row w comes from the row's source offset.
__global__ __launch_bounds__(256) void repack_rows_kernel(RepackDesc r, int64_t rows, int cpr, int es) {
    const int64_t total = rows * cpr;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        const int64_t w = i / cpr;
        const int c = (int)(i - w * cpr);
        const char* s = static_cast<const char*>(r.src) + outer_offset(r, r.ndim - 1, w) * es + (int64_t)c * 16;
        *reinterpret_cast<u32x4*>(static_cast<char*>(r.dst) + i * 16) = *reinterpret_cast<const u32x4*>(s);
    }
}

// dst[o][i][j] = src[outer(o) + i + j * sC]: tiles of 64 (i) x 64 (j) elements.  Loads: lane l of a
// tile row reads i = i0 + l % 64 (contiguous in the source); stores: lane l writes j = j0 + l % 64
// (contiguous in the destination).  The LDS tile is padded by one element per row.
template <typename E>
__global__ __launch_bounds__(256) void repack_transpose_kernel(RepackDesc r, int64_t tiles_i, int64_t tiles_j) {
    __shared__ E tile[64][65];
    const int nd = r.ndim;
    const int64_t R = r.shape[nd - 2], C = r.shape[nd - 1], sC = r.strides[nd - 1];
    const int64_t per_outer = tiles_i * tiles_j;
    const int64_t total = per_outer * (r.numel / (R * C));
    const int l = threadIdx.x & 63, q = threadIdx.x >> 6;
    const E* src = static_cast<const E*>(r.src);
    E* dst = static_cast<E*>(r.dst);
    for (int64_t t = blockIdx.x; t < total; t += gridDim.x) {
        const int64_t o = t / per_outer;
        const int64_t rem = t - o * per_outer;
        const int64_t i0 = (rem / tiles_j) * 64, j0 = (rem % tiles_j) * 64;
        const int64_t base = outer_offset(r, nd - 2, o);
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const int jj = q + 4 * k;
            if (i0 + l < R && j0 + jj < C) tile[jj][l] = src[base + (i0 + l) + (j0 + jj) * sC];
        }
        __syncthreads();
        E* out = dst + o * R * C;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const int ii = q + 4 * k;
            if (i0 + ii < R && j0 + l < C) out[(i0 + ii) * C + j0 + l] = tile[l][ii];
        }
        __syncthreads();
    }
}

// 16-bit elements moved in pairs: the same tiles, with 4-byte loads of two consecutive i and 4-byte
// stores of two consecutive j.  Requires even R and C, even outer strides and 4-byte aligned
// buffers (checked by the launcher), so every pair lies inside the view and is aligned.
__global__ __launch_bounds__(256) void repack_transpose16_kernel(RepackDesc r, int64_t tiles_i, int64_t tiles_j) {
    __shared__ uint16_t tile[64][66];
    const int nd = r.ndim;
    const int64_t R = r.shape[nd - 2], C = r.shape[nd - 1], sC = r.strides[nd - 1];
    const int64_t per_outer = tiles_i * tiles_j;
    const int64_t total = per_outer * (r.numel / (R * C));
    const int p = threadIdx.x & 31, q = threadIdx.x >> 5; // pair index, row group (8)
    const uint16_t* src = static_cast<const uint16_t*>(r.src);
    uint16_t* dst = static_cast<uint16_t*>(r.dst);
    for (int64_t t = blockIdx.x; t < total; t += gridDim.x) {
        const int64_t o = t / per_outer;
        const int64_t rem = t - o * per_outer;
        const int64_t i0 = (rem / tiles_j) * 64, j0 = (rem % tiles_j) * 64;
        const int64_t base = outer_offset(r, nd - 2, o);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int jj = q + 8 * k;
            if (i0 + 2 * p < R && j0 + jj < C) {
                const unsigned v = *reinterpret_cast<const unsigned*>(src + base + (i0 + 2 * p) + (j0 + jj) * sC);
                tile[jj][2 * p] = (uint16_t)(v & 0xFFFFu);
                tile[jj][2 * p + 1] = (uint16_t)(v >> 16);
            }
        }
        __syncthreads();
        uint16_t* out = dst + o * R * C;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int ii = q + 8 * k;
            if (i0 + ii < R && j0 + 2 * p < C) {
                const unsigned v = (unsigned)tile[2 * p][ii] | ((unsigned)tile[2 * p + 1][ii] << 16);
                *reinterpret_cast<unsigned*>(out + (i0 + ii) * C + j0 + 2 * p) = v;
            }
        }
        __syncthreads();
    }
}

static unsigned grid_for(int64_t items, int64_t per_block) {
    int64_t blocks = (items + per_block - 1) / per_block;
    if (blocks > 65536) blocks = 65536;
    return (unsigned)(blocks < 1 ? 1 : blocks);
}

template <typename E>
static int launch_transpose(const RepackDesc& r, hipStream_t stream) {
    const int nd = r.ndim;
    const int64_t R = r.shape[nd - 2], C = r.shape[nd - 1];
    const int64_t tiles_i = (R + 63) / 64, tiles_j = (C + 63) / 64;
    const int64_t total = tiles_i * tiles_j * (r.numel / (R * C));
    if constexpr (sizeof(E) == 2) {
        bool pairs = R % 2 == 0 && C % 2 == 0 && r.strides[nd - 1] % 2 == 0 &&
                     (reinterpret_cast<uintptr_t>(r.src) % 4) == 0 && (reinterpret_cast<uintptr_t>(r.dst) % 4) == 0;
        for (int d = 0; d < nd - 2; ++d)
            if (r.shape[d] > 1 && r.strides[d] % 2 != 0) pairs = false;
        if (pairs) {
            hipLaunchKernelGGL(repack_transpose16_kernel, dim3(grid_for(total, 1)), dim3(256), 0, stream, r, tiles_i, tiles_j);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL(repack_transpose_kernel<E>, dim3(grid_for(total, 1)), dim3(256), 0, stream, r, tiles_i, tiles_j);
    return hipGetLastError();
}

// Zero-padded row copies of a GEMM's operands (pad_gemm_operands uses them for operands contiguous
// along one dimension whose rows are not whole 16-byte chunks): destination row w = batch * rows + row
// holds the source row's L elements, then zeros up to P.  One thread per 16-byte destination chunk,
// consecutive threads on consecutive chunks (rows run on one after the other).  A chunk wholly inside
// its row is one 16-byte load, at whatever alignment the row has (global loads here need none beyond
// the byte): element by element, 16 loads per int8 chunk, the copy took longer than the product it
// fed.  Both operands' copies are one launch,
// the first `blocks_a` workgroups for the first: a launch more costs 3 to 4 us.
// Whole calls, us: int8 [3,3695]@Wt[3695,2496] 24.0 -> 14.9, bf16 [2,2277]@Wt[2277,2238] 20.2 -> 15.7,
// int8 [512,590]@Bt[590,448] 10.5 -> 7.4, bf16 [209,3794]@[3794,2284] 41.8 -> 37.0.
// IDX: 32-bit index arithmetic when the chunk count allows.
template <typename E, typename IDX>
__device__ inline void pad_rows(const PadJob& j, IDX first, IDX stride) {
    constexpr int V = 16 / (int)sizeof(E);
    struct Chunk {
        E e[V];
    };
    const IDX cpr = (IDX)(j.P / V);
    const IDX total = (IDX)j.nrows * cpr;
    const IDX rws = (IDX)j.rows;
    for (IDX i = first; i < total; i += stride) {
        const IDX w = i / cpr, c = i - w * cpr;
        const IDX b = rws == (IDX)j.nrows ? 0 : w / rws, r = w - b * rws;
        const E* s = static_cast<const E*>(j.src) + (int64_t)b * j.s_batch + (int64_t)r * j.s_row;
        const int64_t x0 = (int64_t)c * V;
        u32x4 v;
        if (j.L >= V) { // uniform
            // The row's last 16 bytes serve its partial chunk, shifted down (zeros follow).
            const int64_t x = x0 + V <= j.L ? x0 : j.L - V;
            unsigned __int128 q;
            __builtin_memcpy(&q, reinterpret_cast<const char*>(s + x), 16);
            q >>= (unsigned)(x0 - x) * 8 * (unsigned)sizeof(E);
            v = __builtin_bit_cast(u32x4, q);
        } else {
            Chunk t;
#pragma unroll
            for (int e = 0; e < V; ++e) t.e[e] = x0 + e < j.L ? s[x0 + e] : E(0);
            v = __builtin_bit_cast(u32x4, t);
        }
        *reinterpret_cast<u32x4*>(static_cast<E*>(j.dst) + (int64_t)w * j.P + x0) = v;
    }
}
template <typename E, typename IDX>
__global__ __launch_bounds__(256) void pad_rows_kernel(PadJob a, PadJob b, unsigned blocks_a) {
    if (blockIdx.x < blocks_a) pad_rows<E, IDX>(a, (IDX)blockIdx.x * 256 + threadIdx.x, (IDX)blocks_a * 256);
    else pad_rows<E, IDX>(b, (IDX)(blockIdx.x - blocks_a) * 256 + threadIdx.x, (IDX)(gridDim.x - blocks_a) * 256);
}

int launch_pad_rows(const PadJob* jobs, int n, int es, hipStream_t stream) {
    if (n < 1 || n > 2) return TV_E_SHAPE;
    unsigned blocks[2] = {0, 0};
    bool small = true;
    for (int i = 0; i < n; ++i) {
        const PadJob& j = jobs[i];
        if (j.nrows <= 0 || j.L <= 0 || j.P < j.L || (j.P * es) % 16 != 0) return TV_E_SHAPE;
        const int64_t chunks = j.nrows * (j.P * es / 16);
        blocks[i] = grid_for(chunks, 256);
        small = small && chunks < ((int64_t)1 << 31);
    }
    const PadJob& b = jobs[n - 1];
    const dim3 grid(blocks[0] + blocks[1]);
#define TV_PAD(E)                                                                                                      \
    if (small) hipLaunchKernelGGL((pad_rows_kernel<E, uint32_t>), grid, dim3(256), 0, stream, jobs[0], b, blocks[0]);  \
    else hipLaunchKernelGGL((pad_rows_kernel<E, int64_t>), grid, dim3(256), 0, stream, jobs[0], b, blocks[0]);
    switch (es) {
        case 1: TV_PAD(uint8_t) break;
        case 2: TV_PAD(uint16_t) break;
        case 4: TV_PAD(uint32_t) break;
        default: return TV_E_DTYPE;
    }
#undef TV_PAD
    return hipGetLastError();
}

int launch_repack(const tv_repack_args* a, hipStream_t stream) {
    RepackDesc r;
    r.ndim = a->ndim;
    r.numel = 1;
    for (int d = 0; d < a->ndim; ++d) {
        r.shape[d] = a->shape[d];
        r.strides[d] = a->strides[d];
        r.numel *= a->shape[d];
    }
    r.src = a->src;
    r.dst = a->dst;
    if (r.numel == 0) return 0;
    const int es = a->elem_size;
    if (es != 1 && es != 2 && es != 4 && es != 8) return TV_E_DTYPE;
    const int nd = r.ndim;

    // Rows: contiguous innermost dimension in whole, aligned 16-byte chunks.
    if (nd >= 1 && r.strides[nd - 1] == 1 && (r.shape[nd - 1] * es) % 16 == 0 &&
        (reinterpret_cast<uintptr_t>(r.src) % 16) == 0 && (reinterpret_cast<uintptr_t>(r.dst) % 16) == 0) {
        bool aligned = true;
        for (int d = 0; d < nd - 1; ++d)
            if (r.shape[d] > 1 && (r.strides[d] * es) % 16 != 0) aligned = false;
        const int64_t cpr = r.shape[nd - 1] * es / 16;
        if (aligned && cpr <= 0x7FFFFFFF) {
            const int64_t rows = r.numel / r.shape[nd - 1];
            hipLaunchKernelGGL(repack_rows_kernel, dim3(grid_for(rows * cpr, 256)), dim3(256), 0, stream, r, rows, (int)cpr, es);
            return hipGetLastError();
        }
    }
    // Transpose of the last two dimensions.
    if (nd >= 2 && r.strides[nd - 2] == 1 && r.strides[nd - 1] != 1 && r.shape[nd - 2] > 1 && r.shape[nd - 1] > 1) {
        switch (es) {
            case 1: return launch_transpose<uint8_t>(r, stream);
            case 2: return launch_transpose<uint16_t>(r, stream);
            case 4: return launch_transpose<uint32_t>(r, stream);
            default: return launch_transpose<uint64_t>(r, stream);
        }
    }
    const unsigned blocks = grid_for(r.numel, 256);
    switch (es) {
        case 1: hipLaunchKernelGGL(repack_kernel<uint8_t>, dim3(blocks), dim3(256), 0, stream, r); break;
        case 2: hipLaunchKernelGGL(repack_kernel<uint16_t>, dim3(blocks), dim3(256), 0, stream, r); break;
        case 4: hipLaunchKernelGGL(repack_kernel<uint32_t>, dim3(blocks), dim3(256), 0, stream, r); break;
        default: hipLaunchKernelGGL(repack_kernel<uint64_t>, dim3(blocks), dim3(256), 0, stream, r); break;
    }
    return hipGetLastError();
}

} // namespace tvk
