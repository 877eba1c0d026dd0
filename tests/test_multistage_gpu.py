"""The multi-stage direct-load GEMM (gemm_ms_impl.h) at the edges of its tiles, its k-stages and its
split ranges, exact: integer inputs in [-3, 3] make every order of summation give the same fp32 / int32
sums, so the results equal numpy's product rounded once (int8: its low byte), bit for bit.

The shapes take the tiles of up to 64 rows whole and split (at 16 bits 32x64 and 64x64, in int8 64x128 as well),
the two-stage 128x128 tiles and, in fp32, the split two-stage tiles, with ragged M, N and K (fewer k-tiles than stages;
one element past a k-tile), M-contiguous and K-contiguous operands, batches, rotated k-loops (many rows of A, one
tile column) and the fused epilogue.  Each instantiation at its edges, the 128x128 and 256x128 multi-stage tiles
and the rotated 256x128 tile among them: tests/test_kernel_cases_gpu.py.
"""
import ctypes

import numpy as np
import pytest
import torch

from tensorvia_amd import rng
from tests.util import BFLOAT16, FLOAT16, FLOAT32, INT8, to_storage, to_torch

pytestmark = pytest.mark.gpu

# (M, N, K): 16-byte rows in every dtype and layout, so no padded copies.
SHAPES = [(16, 64, 16), (32, 64, 144), (48, 1216, 3712), (64, 64, 8192), (96, 2048, 1040), (128, 4096, 2048), (272, 528, 336),
          (528, 2064, 1040), (1024, 1040, 528), (2064, 1040, 272), (336, 11008, 1024)]
TALL = [(8192, 128, 1024), (8208, 64, 1040), (4112, 112, 2048)]
DTYPES = [FLOAT32, BFLOAT16, FLOAT16, INT8]


def _ints(seed, shape):
    return rng.uniform_int(seed, int(np.prod(shape)), -3, 3).reshape(shape)


def _enc(x, dt):
    if dt == INT8:
        return x.astype(np.int64).astype(np.int8)
    x = x.astype(np.float32)
    return rng.f32_to_bf16_bits(x) if dt == BFLOAT16 else rng.f32_to_f16_bits(x) if dt == FLOAT16 else x


def _dev(x, dt, trans):
    if trans:
        return to_torch(np.ascontiguousarray(_enc(np.swapaxes(x, -1, -2), dt)), dt).transpose(-1, -2)
    return to_torch(np.ascontiguousarray(_enc(x, dt)), dt)


def _check(hip, dt, x, y, at, bt):
    c = hip.gemm(_dev(x, dt, at), _dev(y, dt, bt))
    torch.cuda.synchronize()
    np.testing.assert_array_equal(to_storage(c), _enc(np.matmul(x.astype(np.float64), y.astype(np.float64)), dt))


@pytest.mark.parametrize("dt", DTYPES, ids=["fp32", "bf16", "fp16", "int8"])
@pytest.mark.parametrize("at,bt", [(False, False), (False, True), (True, False), (True, True)], ids=["kn", "nk", "At-kn", "At-nk"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_tiles_and_splits_exact(hip, dt, at, bt, shape):
    M, N, K = shape
    _check(hip, dt, _ints(M + K, (M, K)), _ints(N + K, (K, N)), at, bt)


@pytest.mark.parametrize("dt", DTYPES, ids=["fp32", "bf16", "fp16", "int8"])
@pytest.mark.parametrize("shape", TALL, ids=lambda s: "x".join(map(str, s)))
def test_rotated_exact(hip, dt, shape):
    M, N, K = shape
    _check(hip, dt, _ints(M + K, (M, K)), _ints(N + K, (K, N)), False, False)
    B = 4  # the same rows as a batch: each entry its own B
    x, y = _ints(M + K, (B, M // B // 16 * 16, K)), _ints(N + K, (B, K, N))
    _check(hip, dt, x, y, False, False)


@pytest.mark.parametrize("dt", [FLOAT32, BFLOAT16, INT8], ids=["fp32", "bf16", "int8"])
def test_repeated_and_noalloc_exact(hip, dt):
    """A split call leaves its counters at zero (ten calls, other shapes between); the entry point
    without a workspace runs unsplit."""
    lib = hip.lib()
    sh = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    cases = []
    for M, N, K in [(48, 1216, 3712), (64, 64, 8192), (80, 2048, 2064)]:
        x, y = _ints(M, (M, K)), _ints(N, (K, N))
        tx, ty = _dev(x, dt, False), _dev(y, dt, True)
        cases.append((tx, ty, _enc(np.matmul(x.astype(np.float64), y.astype(np.float64)), dt)))
    for _ in range(10):
        for tx, ty, want in cases:
            np.testing.assert_array_equal(to_storage(hip.gemm(tx, ty)), want)
    for tx, ty, want in cases:
        c = torch.empty((tx.shape[0], ty.shape[1]), dtype=tx.dtype, device="cuda")
        hip.check(lib.tv_hip_gemm_noalloc(ctypes.byref(hip.make_args(tx, ty, c)), sh))
        torch.cuda.synchronize()
        np.testing.assert_array_equal(to_storage(c), want)


@pytest.mark.parametrize("dt", [FLOAT32, BFLOAT16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("shape", [(48, 1216, 3712), (272, 528, 336), (336, 11008, 1024), (4112, 112, 2048)],
                         ids=lambda s: "x".join(map(str, s)))
def test_fused_relu_bias_exact(hip, dt, shape):
    M, N, K = shape
    x, y, bias = _ints(M, (M, K)), _ints(N, (K, N)), _ints(K, (N,))
    want = _enc(np.maximum(np.matmul(x.astype(np.float64), y.astype(np.float64)) + bias, 0), dt)
    tx, ty, tb = _dev(x, dt, False), _dev(y, dt, False), _dev(bias, dt, False)
    c = torch.empty((M, N), dtype=tx.dtype, device="cuda")
    ep = hip.TvEpilogue()
    ep.act, ep.bias, ep.sbias_n = hip.ACT_RELU, tb.data_ptr(), 1
    hip.check(hip.lib().tv_hip_gemm_ex(ctypes.byref(hip.make_args(tx, ty, c)), ctypes.byref(ep),
                                       ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    np.testing.assert_array_equal(to_storage(c), want)


@pytest.mark.parametrize("dt", DTYPES, ids=["fp32", "bf16", "fp16", "int8"])
@pytest.mark.parametrize("shape", [(40, 67, 64), (130, 257, 192), (520, 1031, 256), (2064, 1029, 128), (4096, 2047, 64)],
                         ids=lambda s: "x".join(map(str, s)))
def test_unaligned_rows_of_c_exact(hip, dt, shape):
    """C rows at any alignment (odd N; a start inside wider rows): every element stored, none beside."""
    M, N, K = shape
    x, y = _ints(M, (M, K)), _ints(N, (K, N))
    want = _enc(np.matmul(x.astype(np.float64), y.astype(np.float64)), dt)
    tx, ty = _dev(x, dt, False), _dev(y, dt, True)
    for pad, off in ((0, 0), (3, 1), (16, 5)):
        wide = torch.full((M, N + pad), 77, dtype=tx.dtype, device="cuda")
        hip.gemm(tx, ty, out=wide[:, off:off + N])
        torch.cuda.synchronize()
        np.testing.assert_array_equal(to_storage(wide[:, off:off + N].contiguous()), want)
        assert bool((wide[:, :off] == 77).all()) and bool((wide[:, off + N:] == 77).all())


TINY = [(1, 1, 1), (9, 15, 1), (16, 16, 128), (17, 33, 129), (31, 128, 33), (128, 128, 128), (129, 16, 64), (9, 1, 127)]


@pytest.mark.parametrize("dt", DTYPES, ids=["fp32", "bf16", "fp16", "int8"])
@pytest.mark.parametrize("shape", TINY, ids=lambda s: "x".join(map(str, s)))
def test_smallest_products_exact(hip, dt, shape):
    """The 16 x 16-block kernel of the smallest products, its edges and one past its limits: row-major,
    transposed and column-stepped operands, batches, a column-strided C."""
    M, N, K = shape
    x, y = _ints(M + K, (3, M, K)), _ints(N + K, (3, K, N))
    want = _enc(np.matmul(x.astype(np.float64), y.astype(np.float64)), dt)
    for at in (False, True):
        for bt in (False, True):
            np.testing.assert_array_equal(to_storage(hip.gemm(_dev(x, dt, at), _dev(y, dt, bt))), want)
    wide = np.zeros((3, M, 2 * K), x.dtype)
    wide[..., ::2] = x
    np.testing.assert_array_equal(to_storage(hip.gemm(_dev(wide, dt, False)[..., ::2], _dev(y, dt, False))), want)
    c = torch.zeros((3, N, M), dtype=_dev(x[:1], dt, False).dtype, device="cuda").transpose(1, 2)
    hip.gemm(_dev(x, dt, False), _dev(y, dt, False), out=c)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(to_storage(c.contiguous()), want)


@pytest.mark.parametrize("dt", DTYPES, ids=["fp32", "bf16", "fp16", "int8"])
@pytest.mark.parametrize("K", [31, 32, 33, 48, 63, 64, 65, 128])
def test_smallest_products_by_k_exact(hip, dt, K):
    """Each of the 16 x 16-block kernel's instantiations (up to 32, 64 and 128 k) at its edges, aligned and
    unaligned rows, more blocks than CUs."""
    for B, M, N in ((1, 17, 48), (1, 33, 47), (40, 20, 96)):
        x, y = _ints(M + K, (B, M, K)), _ints(N + K, (B, K, N))
        want = _enc(np.matmul(x.astype(np.float64), y.astype(np.float64)), dt)
        for at, bt in ((False, False), (False, True), (True, False)):
            np.testing.assert_array_equal(to_storage(hip.gemm(_dev(x, dt, at), _dev(y, dt, bt))), want)


@pytest.mark.parametrize("dt", [FLOAT32, BFLOAT16, INT8], ids=["fp32", "bf16", "int8"])
@pytest.mark.parametrize("shape", [(64, 64, 8192), (48, 1216, 3712), (65, 77, 2049)], ids=lambda s: "x".join(map(str, s)))
def test_cold_capture_exact(hip, dt, shape):
    """A call that wants a workspace, captured on a stream that has none yet: the captured call runs
    without it, and every replay gives the exact result, eager calls of the same shape between."""
    M, N, K = shape
    x, y = _ints(M, (M, K)), _ints(N, (K, N))
    want = _enc(np.matmul(x.astype(np.float64), y.astype(np.float64)), dt)
    tx, ty = _dev(x, dt, False), _dev(y, dt, True)
    out = torch.zeros((M, N), dtype=tx.dtype, device="cuda")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=torch.cuda.Stream()):
        hip.gemm(tx, ty, out=out)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(to_storage(out), want)
        np.testing.assert_array_equal(to_storage(hip.gemm(tx, ty)), want)
