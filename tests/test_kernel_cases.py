"""The calls of tests/kernel_cases.py launch the kernels they are listed with (no GPU)."""
import pytest

from tests.kernel_cases import CASES, TYPE_NAMES
from tests.routes import call, run
from tests.util import BFLOAT16, FLOAT16


@pytest.mark.parametrize("dt", list(CASES) + [FLOAT16])
def test_each_call_launches_its_kernel(dt):
    cases = CASES[BFLOAT16 if dt == FLOAT16 else dt]
    lines = [call(M, K, N, dt, batch=b, at=bool(at), bt=bool(bt), act=act, bias=act) for _, _, (b, M, K, N), at, bt, act in cases]
    wrong = []
    for (kernel, split, (b, M, K, N), *_), r in zip(cases, run(*lines)):
        kernel = kernel.replace("<T,", f"<{'_Float16' if dt == FLOAT16 else TYPE_NAMES[dt]},")
        bm, bn = (int(x) for x in kernel.split(",")[1:3])
        tiles = b * -(-M // bm) * -(-N // bn)
        got_split = r.kernel.startswith("gemm_ms") and r.launches[-1][1] != tiles
        if r.rc or r.kernel != kernel or got_split != bool(split):
            wrong.append((kernel, split, (b, M, K, N), r.launches))
    assert not wrong, wrong
