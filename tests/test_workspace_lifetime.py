"""The per-stream workspace and captured graphs, on the recorded runtime (no GPU): a buffer whose address a
capture recorded is neither freed nor given to an eager call afterwards, whatever later calls need."""
import pytest

from tests.routes import call, run
from tests.util import BFLOAT16, FLOAT32

# Each user of the workspace: a call, and a larger one of the same kind.
USERS = {
    "split_tiles": (call(48, 3712, 1216, BFLOAT16, bt=True), call(333, 4096, 11008, BFLOAT16)),
    "fp32_stream_k": (call(300, 4096, 4096, FLOAT32), call(2592, 2048, 4096, FLOAT32)),
    "gemv_split_k": (call(1, 4096, 4096, BFLOAT16), call(8, 32768, 19200, BFLOAT16)),
    "padded_copies": (call(64, 700, 260, BFLOAT16), call(4096, 4095, 4097, BFLOAT16)),
}


def _ids(results, kind):
    return [i for r in results for i in r.ids(kind)]


@pytest.mark.parametrize("user", USERS)
def test_recorded_buffers_stay(user):
    small, large = USERS[user]
    warm, captured, *later = run(small, "capture 1", small, "capture 0", small, large, large, "capture 1", small, large, "capture 0", large)
    recorded = warm.ids("malloc")
    assert recorded, "the call holds no workspace"
    assert not captured.ids("malloc") and captured.launches == warm.launches
    assert all(r.rc == 0 for r in (warm, captured, *later))
    assert not set(recorded) & set(_ids(later, "free")), "a buffer that a graph recorded was freed"
    # The eager call after the capture has buffers of its own; the graph's are not shared with it.
    assert len(later[0].ids("malloc")) == len(recorded)
    # The second capture takes the large call's buffers over; the eager call after it allocates again.
    assert not _ids(later[3:5], "malloc") and later[5].ids("malloc")
    assert not any(e[0].startswith("illegal") for r in (warm, captured, *later) for e in r.events)


def test_capture_without_a_warm_up_holds_nothing():
    for small, large in USERS.values():
        cold, = run("capture 1", large)
        assert cold.rc == 0 and cold.launches
        assert not cold.ids("malloc") and not any(e[0].startswith("illegal") for e in cold.events)


def test_buffers_of_ever_larger_captures_are_bounded():
    """Graphs captured for ever larger calls: what stays allocated is at most eight times the last buffer."""
    lines = []
    for m in range(1100, 4200, 60):
        c = call(m, 4095, 4097, BFLOAT16)
        lines += [c, "capture 1", c, "capture 0"]
    live = {}
    for r in run(*lines):
        for e in r.events:
            if e[0] == "malloc":
                live[int(e[1])] = int(e[2])
            elif e[0] == "free":
                live.pop(int(e[1]))
    per_kind = sorted(live.values())
    assert sum(per_kind) <= 8 * 2 * per_kind[-1]


def test_a_failed_rounded_allocation_is_asked_for_exactly():
    """A[4100, 4095] in rows of 4096: 40 MiB rounded, 4100 x 4096 x 2 bytes where that fails."""
    r, = run("fail 1", call(4100, 4095, 4097, BFLOAT16))
    failed = [int(e[1]) for e in r.events if e[0] == "malloc-failed"]
    got = [int(e[2]) for e in r.events if e[0] == "malloc"]
    assert r.rc == 0 and failed == [40 << 20] and got[0] == 4100 * 4096 * 2


def test_the_gpu_suites_cases_use_the_workspace():
    """The calls that tests/test_workspace_gpu.py and tests/test_concurrency_gpu.py run as users of the workspace."""
    from tests.test_concurrency_gpu import CASES as threads
    from tests.test_workspace_gpu import CASES as memory
    calls = [(n, call(*sa, sb[1], dt)) for n, dt, sa, sb, _ in memory] + [(n, call(M, K, N, dt)) for n, dt, M, K, N, _ in threads]
    for name, line in calls:
        r, = run(line)
        assert bool(r.ids("malloc")) == (name not in ("fp32_stream_k", "int8_stream_k")), name
