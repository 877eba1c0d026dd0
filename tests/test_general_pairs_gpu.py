"""The kernels of the dtype pairs without 8/16/32-bit matrix-core types (gemm_simt.hip, gemm_f64.hip): tiles
at the edges of their 64- and 32-wide tiles, 32-wide k-steps and 64-wide k-chunks, and a thread per output,
against the oracle's MulImpl<CPU>: row-major, transposed and strided views, batches, broadcast.

Integer pairs equal the oracle bit for bit, wrap-around included.  Float pairs sum the same products
in the oracle's order up to the fusing of a multiply and an add, so each output differs by at most
two roundings per term: |c - ref| <= 2 K eps sum |a| |b|.
"""
import numpy as np
import pytest
import torch

import oracle as orc
from tests.util import BFLOAT16, FLOAT16, FLOAT32, to_storage, to_torch
from tensorvia_amd import rng

pytestmark = pytest.mark.gpu

I8, I16, I32, I64, F64 = 0, 1, 2, 3, 7
INT_LIM = {I8: 100, I16: 30000, I32: 2**30, I64: 2**61}
PAIRS = [(F64, F64), (FLOAT32, BFLOAT16), (FLOAT16, FLOAT32), (BFLOAT16, FLOAT16), (FLOAT32, F64), (I16, I16), (I32, I32),
         (I16, I32), (I8, I64)]
SHAPES = [(1, 1, 1), (31, 63, 33), (64, 64, 64), (65, 97, 63), (33, 32, 130), (200, 129, 300)]
# The calls above run a thread per output but for the last; these run on tiles (test_routes.py), 64 x 64 and, in
# fp64, 32 x 32 up to 191 of the large ones.
TILED = [(577, 97, 513), (897, 97, 897), (705, 129, 641), (640, 31, 832), (833, 64, 639)]
LARGE = [(1030, 97, 1021), (1024, 64, 1024)]  # 2^20 outputs and more: 64-wide chunk sums


def _values(seed, shape, dt):
    r = np.random.default_rng(seed)
    if dt <= I64:
        return r.integers(-INT_LIM[dt], INT_LIM[dt], shape).astype(orc.NP[dt])
    x = r.uniform(-1, 1, shape)
    if dt == F64:
        return x
    x = x.astype(np.float32)
    return rng.f32_to_bf16_bits(x) if dt == BFLOAT16 else rng.f32_to_f16_bits(x) if dt == FLOAT16 else x


def _f64(x, dt):
    return (rng.bf16_bits_to_f32(x) if dt == BFLOAT16 else rng.f16_bits_to_f32(x) if dt == FLOAT16 else x).astype(np.float64)


def _view(x, dt, layout):
    if layout == "trans":
        return to_torch(np.ascontiguousarray(np.swapaxes(x, -1, -2)), dt).transpose(-1, -2)
    if layout == "step":  # every other column, every third row of a larger tensor
        big = np.zeros(x.shape[:-2] + (3 * x.shape[-2], 2 * x.shape[-1]), dtype=x.dtype)
        big[..., ::3, ::2] = x
        return to_torch(big, dt)[..., ::3, ::2]
    return to_torch(np.ascontiguousarray(x), dt)


def _check(hip, da, db, a, b, ta, tb):
    rt = orc.result_type(da, db)
    got = to_storage(hip.gemm(ta, tb, out_dtype=rt))
    ref = np.stack([orc.mul(a[i], da, b[i] if b.ndim == 3 else b, db) for i in range(a.shape[0])]) if a.ndim == 3 else orc.mul(a, da, b, db)
    if ref.dtype.kind != "f":
        np.testing.assert_array_equal(got, ref)
        return
    x, y = np.abs(_f64(a, da)), np.abs(_f64(b, db))
    # The type the products and sums run in may be the narrower one (A's type in the chunked sums).
    eps = 2.0**-23 if FLOAT32 in (da, db) or F64 not in (da, db) else 2.0**-52
    bound = 2 * a.shape[-1] * eps * np.matmul(x, y)
    assert bool((np.abs(got.astype(np.float64) - ref.astype(np.float64)) <= bound).all())


@pytest.mark.parametrize("pair", PAIRS, ids=lambda p: f"{p[0]}x{p[1]}")
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_general_pairs_edges(hip, pair, shape):
    (da, db), (M, K, N) = pair, shape
    a, b = _values(M + 3 * K, (M, K), da), _values(N + 5 * K, (K, N), db)
    for la, lb in (("row", "row"), ("row", "trans"), ("trans", "row"), ("step", "step")):
        _check(hip, da, db, a, b, _view(a, da, la), _view(b, db, lb))


@pytest.mark.parametrize("pair", PAIRS, ids=lambda p: f"{p[0]}x{p[1]}")
@pytest.mark.parametrize("shape", TILED, ids=lambda s: "x".join(map(str, s)))
def test_general_pairs_tile_edges(hip, pair, shape):
    (da, db), (M, K, N) = pair, shape
    a, b = _values(M + 3 * K, (M, K), da), _values(N + 5 * K, (K, N), db)
    for la, lb in (("row", "row"), ("trans", "trans"), ("step", "step")):
        _check(hip, da, db, a, b, _view(a, da, la), _view(b, db, lb))


@pytest.mark.parametrize("pair", PAIRS, ids=lambda p: f"{p[0]}x{p[1]}")
@pytest.mark.parametrize("shape", LARGE, ids=lambda s: "x".join(map(str, s)))
def test_general_pairs_chunked(hip, pair, shape):
    (da, db), (M, K, N) = pair, shape
    a, b = _values(M + 3 * K, (M, K), da), _values(N + 5 * K, (K, N), db)
    _check(hip, da, db, a, b, _view(a, da, "row"), _view(b, db, "trans"))


@pytest.mark.parametrize("pair", [(F64, F64), (FLOAT32, BFLOAT16), (I32, I32)], ids=lambda p: f"{p[0]}x{p[1]}")
def test_general_pairs_batched(hip, pair):
    da, db = pair
    a, b, b1 = _values(1, (3, 70, 45), da), _values(2, (3, 45, 66), db), _values(3, (45, 66), db)
    _check(hip, da, db, a, b, _view(a, da, "row"), _view(b, db, "row"))
    _check(hip, da, db, a, b1, _view(a, da, "step"), _view(b1, db, "trans"))


@pytest.mark.parametrize("pair", PAIRS, ids=lambda p: f"{p[0]}x{p[1]}")
def test_general_pairs_small_matrices(hip, pair):
    """Batches of small matrices and thin ones, a thread per output: every remainder of its groups of 8 k, views,
    broadcast operands, a column-strided C."""
    da, db = pair
    for B, M, K, N in ((300, 4, 5, 3), (64, 1, 130, 1), (40, 5, 71, 7), (200, 3, 8, 9), (90, 2, 1, 2)):
        a, b = _values(M + 3 * K, (B, M, K), da), _values(N + 5 * K, (B, K, N), db)
        for la, lb in (("row", "row"), ("trans", "trans"), ("step", "step")):
            _check(hip, da, db, a, b, _view(a, da, la), _view(b, db, lb))
        _check(hip, da, db, a, b[0], _view(a, da, "row"), _view(b[0], db, "trans"))
    a, b = _values(7, (5000, 6), da), _values(8, (6, 3), db)
    _check(hip, da, db, a, b, _view(a, da, "row"), _view(b, db, "row"))
    rt = orc.result_type(da, db)
    c = _view(np.zeros((3, 5000), dtype=orc.NP[rt]), rt, "row").t()
    hip.gemm(_view(a, da, "row"), _view(b, db, "row"), out=c, out_dtype=rt)
    np.testing.assert_array_equal(to_storage(c), to_storage(hip.gemm(_view(a, da, "row"), _view(b, db, "row"), out_dtype=rt)))


@pytest.mark.parametrize("pair", PAIRS, ids=lambda p: f"{p[0]}x{p[1]}")
def test_general_pairs_thin_chunked(hip, pair):
    """2^20 outputs and more with a thread each: 64-wide chunk sums and a last chunk of 3 k."""
    da, db = pair
    a, b = _values(11, (350001, 67), da), _values(12, (67, 3), db)
    _check(hip, da, db, a, b, _view(a, da, "row"), _view(b, db, "row"))
