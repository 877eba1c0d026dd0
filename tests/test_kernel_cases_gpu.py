"""Every GEMM kernel instantiation that the dispatch can choose, at sizes ragged in each tile dimension: the calls
of tests/kernel_cases.py, whose kernels tests/test_kernel_cases.py checks.  Integer inputs in [-2, 2] (sums below
2^24): every order of summation gives the same fp32 / int32 sum, so results equal the 64-bit product rounded once
(int8: its low byte), bit for bit; calls in a row, each after the first with the counters the one before left."""
import ctypes

import pytest
import torch

import tensorvia_amd as tv
from tests.kernel_cases import CASES, case_id
from tests.util import BFLOAT16, FLOAT16, FLOAT32, INT8

pytestmark = pytest.mark.gpu

NAMES = {BFLOAT16: "bf16", FLOAT16: "fp16", FLOAT32: "fp32", INT8: "int8"}


def _run(dt, case, calls=2):
    _, _, (b, M, K, N), at, bt, act = case
    tdt = tv.tv_to_torch(dt)
    g = torch.Generator(device="cuda")
    g.manual_seed(M * 7 + K * 3 + N)

    def operand(rows, cols, trans):
        x = torch.randint(-2, 3, (b, rows, cols), generator=g, device="cuda", dtype=torch.int8)
        return x, (x.transpose(1, 2).contiguous().to(tdt).transpose(1, 2) if trans else x.to(tdt))

    x, a = operand(M, K, at)
    y, w = operand(K, N, bt)
    want = torch.matmul(x.double(), y.double())
    bias = None
    if act:
        bias = torch.randint(-2, 3, (N,), generator=g, device="cuda", dtype=torch.int8)
        want = (want + bias.double()).clamp_(min=0)
        bias = bias.to(tdt)
    want = want.to(torch.int64).to(torch.int8) if dt == INT8 else want.float().to(tdt)
    c = torch.full((b, M, N), 7, dtype=tdt, device="cuda")
    args = tv.make_args(a, w, c)
    ep = tv.TvEpilogue()
    if act:
        ep.act, ep.bias, ep.sbias_n = tv.ACT_RELU, bias.data_ptr(), 1
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for _ in range(calls):
        c.fill_(7)
        tv.check(tv.lib().tv_hip_gemm_ex(ctypes.byref(args), ctypes.byref(ep), s) if act else tv.lib().tv_hip_gemm(ctypes.byref(args), s))
        torch.cuda.synchronize()
        assert torch.equal(c, want)


def _special(dt, case):
    """An infinity in the last row of A and a NaN in the last column of B, both at the last k: the zeros past the
    edges of tiles and k-tiles meet neither, and no other output changes."""
    _, _, (b, M, K, N), at, bt, _ = case
    tdt = tv.tv_to_torch(dt)
    g = torch.Generator(device="cuda")
    g.manual_seed(M + K + N)
    x = torch.randint(-2, 3, (b, M, K), generator=g, device="cuda", dtype=torch.int8)
    y = torch.randint(-2, 3, (b, K, N), generator=g, device="cuda", dtype=torch.int8)
    want = torch.matmul(x.double(), y.double())
    want[:, M - 1, :] = torch.where(y[:, K - 1, :] == 0, float("nan"), y[:, K - 1, :].double().sign() * float("inf"))
    want[:, :, N - 1] = float("nan")
    want = want.float().to(tdt)
    a, w = x.to(tdt), y.to(tdt)
    a[:, M - 1, K - 1] = float("inf")
    w[:, K - 1, N - 1] = float("nan")
    a = a.transpose(1, 2).contiguous().transpose(1, 2) if at else a
    w = w.transpose(1, 2).contiguous().transpose(1, 2) if bt else w
    c = tv.gemm(a, w)
    torch.cuda.synchronize()
    assert bool(((c == want) | (c.isnan() & want.isnan())).all())


@pytest.mark.parametrize("dt,case", [pytest.param(dt, c, id=f"{NAMES[dt]}-{case_id(c)}")
                                     for dt in (BFLOAT16, INT8, FLOAT32) for c in CASES[dt]])
def test_kernel_exact(hip, dt, case):
    _run(dt, case)


@pytest.mark.parametrize("case", [c for i, c in enumerate(CASES[BFLOAT16]) if i % 4 == 0 or "256,128" in c[0]], ids=case_id)
def test_kernel_exact_fp16(hip, case):
    _run(FLOAT16, case)


@pytest.mark.parametrize("dt,case", [pytest.param(dt, c, id=f"{NAMES[dt]}-{case_id(c)}")
                                     for dt in (BFLOAT16, FLOAT32) for c in CASES[dt] if not c[5]])
def test_kernel_special_values(hip, dt, case):
    _special(dt, case)


@pytest.mark.parametrize("dt,case", [pytest.param(dt, c, id=f"{NAMES[dt]}-{case_id(c)}") for dt in (BFLOAT16, INT8, FLOAT32)
                                     for c in CASES[dt] if "mfma" in c[0] and c[5]])
def test_register_staged_kloop_repeated(hip, dt, case):
    """The k-loop that stages its operands through registers, 150 calls of each: a wave one k-tile ahead must not
    store over fragments that another wave has still to read (without that order [6][92,628]@[628,3152] was wrong in one
    fp32 call of forty)."""
    _run(dt, case, 150)
