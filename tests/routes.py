"""The kernels a call launches and what it does to its workspace, without a GPU: libtv_hip.so's host
side on the recorded HIP runtime of tests/cpp/route_driver.cpp (a device of 256 CUs)."""
from __future__ import annotations

import subprocess
from dataclasses import dataclass, field

from tensorvia_amd import build_ext as be
from tests.cpp import build as cpp

ES = (1, 2, 4, 8, 2, 2, 4, 8)  # bytes per element of each dtype


@dataclass
class Result:
    rc: int
    events: list = field(default_factory=list)  # [kind, ...] in order

    @property
    def launches(self):
        """(kernel, grid, block) of the call's launches, the workspace's zero-fills left out."""
        return [(e[1], int(e[2]), int(e[3])) for e in self.events if e[0] == "launch" and e[1] != "gemv_zero_kernel"]

    @property
    def kernel(self):
        """The last launch's kernel: the product's (padded copies come first)."""
        return self.launches[-1][0] if self.launches else None

    def ids(self, kind):
        return [int(e[1]) for e in self.events if e[0] == kind]


def call(M, K, N, dt, out=None, batch=1, at=False, bt=False, shared=False, act=0, bias=0, stream=1, entry="gemm",
         mis=(0, 0, 0), db=None, sa=None, sb=None, sc=None):
    """One call: A[batch, M, K] @ B[batch, K, N] on dense operands (at / bt: transposed views), or on the
    strides given."""
    B = batch if batch > 1 else 0
    sa = sa or ((M * K if B else 0,) + ((1, M) if at else (K, 1)))
    sb = sb or ((0 if shared or not B else K * N,) + ((1, K) if bt else (N, 1)))
    sc = sc or (M * N if B else 0, N, 1)
    v = (dt, dt if db is None else db, dt if out is None else out, batch, M, N, K, *sa, *sb, *sc, stream, act, bias, *mis)
    return entry + " " + " ".join(str(int(x)) for x in v)


def run(*lines):
    """A Result for each call among the lines ("capture 0|1" and "fail N" change the state between)."""
    r = subprocess.run([str(cpp.binary("route_driver")), str(be.KERNEL_LIB)], input="\n".join(lines) + "\n",
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    out, events = [], []
    for line in r.stdout.splitlines():
        e = line.split()
        if e[0] == "rc":
            out.append(Result(int(e[1]), events))
            events = []
        else:
            events.append(e)
    assert not events
    return out
