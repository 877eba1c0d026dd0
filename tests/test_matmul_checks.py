"""The checks of tensorvia_amd.gemm on CPU tensors (the entry point replaced by one that records the descriptor):
the fast path's conditions accept and refuse exactly what _check_shapes does, and the packed descriptor is make_args'
one."""
import ctypes
import importlib
import itertools

import pytest
import torch

import tensorvia_amd as tv
mm = importlib.import_module("tensorvia_amd.matmul")  # the package has a function of that name

SHAPES = [(), (3,), (2, 3), (3, 2), (3, 3), (1, 1), (2, 2, 3), (2, 3, 2), (1, 3, 3), (3, 3, 3), (1, 2, 3, 3)]


@pytest.fixture
def recorded(monkeypatch):
    calls = []
    monkeypatch.setattr(mm, "_entry", lambda name: lambda args, stream: calls.append((name, args, stream)) or 0)
    return calls


@pytest.mark.parametrize("sa,sb", itertools.product(SHAPES, SHAPES))
def test_run_refuses_what_check_shapes_refuses(recorded, sa, sb):
    a, b = torch.zeros(sa), torch.zeros(sb)
    try:
        mm._check_shapes(a, b)
        want = None
    except (RuntimeError, IndexError) as e:
        want = str(e)
    if want is None:
        c = mm.gemm(a, b, stream=5)
        assert c.shape == torch.matmul(a, b).shape and recorded[0][2] == 5
    else:
        with pytest.raises((RuntimeError, IndexError)) as e:
            mm.gemm(a, b, stream=5)
        assert str(e.value) == want and not recorded


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.int8, torch.float64])
def test_packed_descriptor_is_make_args(recorded, dt):
    for sa, sb in (((5, 7), (7, 6)), ((3, 5, 7), (3, 7, 6)), ((3, 5, 7), (7, 6))):
        a = torch.zeros(sa[:-2] + (sa[-1], sa[-2]), dtype=dt).transpose(-1, -2)
        wide = torch.zeros(sb[:-1] + (2 * sb[-1],), dtype=dt)
        for b in (wide[..., ::2], wide[..., 1:1 + sb[-1]]):
            out = torch.zeros(sa[:-1] + (9,), dtype=dt)[..., 2:8]
            assert mm.gemm(a, b, out=out, stream=0) is out
            assert recorded[-1][1] == bytes(ctypes.string_at(ctypes.byref(tv.make_args(a, b, out)), ctypes.sizeof(tv.TvGemmArgs)))


def test_the_current_stream_without_the_private_functions(monkeypatch):
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    assert mm._stream_getter() is mm._public_current_stream
