"""Which kernel, tile and grid a call gets, on the recorded runtime of tests/cpp/route_driver.cpp (no GPU,
256 CUs)."""
import pytest

from tests.routes import call, run
from tests.util import BFLOAT16, FLOAT16, FLOAT32, FLOAT64, INT8, INT16, INT32

SPLIT = {
    "bf16_prompt": dict(M=333, K=4096, N=11008, dt=BFLOAT16),
    "bf16_prompt_fused": dict(M=333, K=4096, N=11008, dt=BFLOAT16, act=2, bias=1),
    "bf16_256x128": dict(M=130, K=8208, N=8000, dt=BFLOAT16),
    "f16_nk": dict(M=48, K=3712, N=1216, dt=FLOAT16, bt=True),
    "int8": dict(M=128, K=4096, N=2048, dt=INT8, bt=True),
    "fp32": dict(M=64, K=8192, N=64, dt=FLOAT32),
    "fp32_nk": dict(M=300, K=2048, N=320, dt=FLOAT32, bt=True),
}


@pytest.mark.parametrize("name", SPLIT)
def test_without_a_workspace_the_call_is_planned_again(name):
    """A call that splits K runs, without room for the slots (under a cold capture, or with allocations
    failing), on the tiles that a plan without a split chooses: tv_hip_gemm_noalloc's."""
    shape = SPLIT[name]
    whole, cold, failed, split = run("fail 0", *([call(**shape, entry="noalloc")] if "act" not in shape else ["fail 1000", call(**shape), "fail 0"]),
                                     "capture 1", call(**shape), "capture 0", "fail 1000", call(**shape), "fail 0", call(**shape))
    assert split.launches[-1] != whole.launches[-1], "the call is not split"
    for r in (cold, failed):
        assert r.rc == 0 and r.launches[-1] == whole.launches[-1]


@pytest.mark.parametrize("shape", [(64, 8192, 64), (300, 2048, 320), (128, 4096, 128), (256, 4096, 256)], ids=str)
def test_fp32_few_long_tiles_without_a_workspace(shape):
    """Unsplit, a 32-row tile of the two-stage kernel takes 22 ns per k whatever its size: the multi-stage tiles
    are cheaper, also where the split two-stage kernel would have been."""
    M, K, N = shape
    for r in run(call(M, K, N, FLOAT32, entry="noalloc"), "capture 1", call(M, K, N, FLOAT32)):
        assert r.rc == 0 and r.kernel.startswith("gemm_ms_kernel<GemmCfg<float")


# fp32 calls that the multi-stage kernel made slower (one or two k-tiles; bound by the output), and ones it serves.
@pytest.mark.parametrize("shape,bt,kernel", [((11, 32, 26480), True, "gemm_mfma_kernel"), ((96, 64, 26512), False, "gemm_mfma_kernel"),
                                             ((25008, 8, 4), False, "gemm_mfma_kernel"), ((43376, 32, 16), True, "gemm_mfma_kernel"),
                                             ((9472, 160, 96), False, "gemm_mfma_kernel"), ((1024, 1024, 1024), False, "gemm_ms_kernel"),
                                             ((128, 4096, 128), False, "gemm_ms_kernel"), ((2592, 2048, 4096), False, "gemm_mfma_sk_kernel"),
                                             ((224, 59008, 460), True, "gemm_ms_kernel<GemmCfg<float,64,64")], ids=str)
def test_fp32_kernel_by_price(shape, bt, kernel):
    M, K, N = shape
    r, = run(call(M, K, N, FLOAT32, bt=bt))
    assert r.rc == 0 and r.kernel.startswith(kernel)


# 16-bit and int8 calls outside the tiles' prices: one row or column of 256x256 tiles, tall streams of A, and
# calls beside each rule's limits.
@pytest.mark.parametrize("M,K,N,kw,kernel", [
    (224, 384, 49184, {}, "256,256"), (256, 1024, 40960, dict(bt=True), "256,256"), (131072, 1152, 256, {}, "256,256"),
    (160, 1024, 160, dict(batch=256), "256,256"), (76512, 880, 176, {}, "128,128"), (131072, 256, 136, {}, "128,128"),
    (2960, 136, 200, dict(batch=56), "128,128"),
    (65536, 2048, 128, {}, "256,128"), (131072, 2048, 72, {}, "256,128"), (65536, 4096, 128, {}, "256,128"),
    (2048, 2048, 128, dict(batch=32), "256,128"), (4096, 2048, 80, dict(batch=16), "128,128"), (50000, 2048, 128, {}, "128,128"),
    (65536, 3072, 96, {}, "128,128"), (131072, 4096, 128, {}, "128,128"), (65536, 2048, 256, {}, "256,256")],
    ids=lambda v: "x".join(f"{a}{b}" for a, b in v.items()) if isinstance(v, dict) else str(v))
def test_tall_and_strip_calls(M, K, N, kw, kernel):
    r, = run(call(M, K, N, BFLOAT16, **kw))
    assert r.rc == 0 and f"GemmCfg<__bf16,{kernel}," in r.kernel
    if (N % 128 == 0 or N == 72) and kernel == "256,128":
        assert r.kernel.startswith("gemm_ms_kernel")


@pytest.mark.parametrize("M,K,N,dt,kernel", [
    (16, 32, 32, FLOAT32, "gemm_tiny_kernel<float,double,32>"), (32, 64, 48, FLOAT32, "gemm_tiny_kernel<float,double,64>"),
    (32, 68, 48, FLOAT32, "gemm_m"), (32, 66, 48, FLOAT32, "gemm_tiny_kernel<float,double,128>"),
    (16, 32, 32, BFLOAT16, "gemm_tiny_kernel<__bf16,float,32>"), (16, 40, 32, BFLOAT16, "gemm_m"),
    (16, 39, 32, BFLOAT16, "gemm_tiny_kernel<__bf16,float,64>"), (40, 64, 32, INT8, "gemm_tiny_kernel<signedchar,int,64>"),
    (40, 80, 32, INT8, "gemm_"), (129, 16, 16, INT8, "gemm_"), (9, 127, 128, FLOAT16, "gemm_tiny_kernel<_Float16,float,128>")], ids=str)
def test_smallest_products(M, K, N, dt, kernel):
    r, = run(call(M, K, N, dt))
    assert r.rc == 0 and r.kernel.startswith(kernel) and ("tiny" in kernel or "tiny" not in r.kernel)


# fp64, integer and mixed pairs: a thread per output where the tiles would be mostly empty.
@pytest.mark.parametrize("M,K,N,dt,kw,kernel", [
    (4, 4, 4, FLOAT64, dict(batch=100000), "gemm_each"), (4, 4, 4, INT32, dict(batch=100000), "gemm_each"),
    (8, 8, 8, INT16, dict(batch=10000), "gemm_each"), (1000000, 3, 3, FLOAT64, {}, "gemm_each"), (4, 5, 3, FLOAT64, dict(batch=300), "gemm_each"),
    (350001, 67, 3, FLOAT64, {}, "gemm_each"), (350001, 67, 3, FLOAT32, dict(db=BFLOAT16), "gemm_each"), (5000, 6, 3, INT32, {}, "gemm_each"),
    (32, 64, 32, FLOAT64, dict(batch=3000), "gemm_f64_kernel<32,"), (40, 64, 40, FLOAT64, dict(batch=3000), "gemm_f64_kernel<64,"),
    (1000, 1000, 1000, FLOAT64, {}, "gemm_f64_kernel<64,"), (200, 300, 129, FLOAT64, {}, "gemm_f64_kernel<32,"),
    (1000, 600, 1000, INT32, {}, "gemm_simt_kernel"), (128, 512, 65, FLOAT32, dict(db=BFLOAT16, bt=True), "gemm_simt_kernel"),
    (512, 600, 512, INT16, {}, "gemm_simt_kernel"), (64, 600, 64, INT16, {}, "gemm_each"),
    (16, 128, 16, INT32, dict(batch=1000), "gemm_each"), (37, 18, 22, INT32, dict(batch=2988), "gemm_each")], ids=str)
def test_general_pairs(M, K, N, dt, kw, kernel):
    for r in run(call(M, K, N, dt, **kw), call(M, K, N, dt, **kw, entry="noalloc")):
        assert r.rc == 0 and r.kernel.startswith(kernel)


def test_general_pairs_tests_run_on_tiles():
    """The shapes that tests/test_general_pairs_gpu.py runs at the edges of the tiles do run on them."""
    from tests.test_general_pairs_gpu import LARGE, PAIRS, TILED
    import oracle as orc
    for da, db in PAIRS:
        for M, K, N in TILED + LARGE:
            for at, bt, step in ((0, 0, 0), (1, 1, 0), (0, 0, 1)):
                st = dict(sa=(0, 3 * 2 * K, 2), sb=(0, 3 * 2 * N, 2)) if step else dict(at=at, bt=bt)
                r, = run(call(M, K, N, da, out=orc.result_type(da, db), db=db, **st))
                assert r.rc == 0 and r.kernel.startswith(("gemm_simt_kernel", "gemm_f64_kernel")), (da, db, M, K, N, r.kernel)
    kernels = {run(call(M, K, N, FLOAT64))[0].kernel for M, K, N in TILED + LARGE}
    assert kernels >= {"gemm_f64_kernel<32,false>", "gemm_f64_kernel<64,false>", "gemm_f64_kernel<64,true>"}


@pytest.mark.parametrize("batch,M,K,N", [(9000000, 64, 200, 64), (20000000, 40, 300, 41), (1, 2146435071, 64, 300), (1, 64, 64, 2146435071),
                                         (8388607, 64, 200, 64)], ids=str)
def test_fp64_calls_larger_than_one_grid(batch, M, K, N):
    """More tiles than one grid holds (2^32 threads): several launches that cover the call."""
    r, = run(call(M, K, N, FLOAT64, batch=batch))
    assert r.rc == 0 and not any(e[0] == "launch-refused" for e in r.events)
    t = 64 if "f64_kernel<64" in r.kernel else 32
    tiles = batch * -(-M // t) * -(-N // t)
    assert sum(grid for _, grid, _ in r.launches) == tiles and all(k == "gemm_f64_kernel<%d,true>" % t for k, _, _ in r.launches)
    assert (len(r.launches) == 1) == (tiles * (512 if t == 64 else 256) < 1 << 32)


@pytest.mark.parametrize("dt", [BFLOAT16, FLOAT16, INT8, FLOAT32], ids=["bf16", "fp16", "int8", "fp32"])
def test_tallest_calls_fit_one_grid(dt):
    """2^31 - 2^20 - 1 rows or columns: tiles whose grid would hold 2^32 threads or more are not chosen."""
    L, lines = 2146435071, []
    for short, K in ((1, 1), (1, 16), (8, 16), (16, 8), (40, 4), (64, 1)):
        for M, N in ((L, short), (short, L))[:2 if short > 32 else 1]:  # up to 32 rows: the GEMV
            for bt in (False, True):
                lines += [call(M, K, N, dt, bt=bt), call(M, K, N, dt, bt=bt, entry="noalloc")]
                if dt != INT8:
                    lines.append(call(M, K, N, dt, bt=bt, act=1))
    for line, r in zip(lines, run(*lines)):
        assert r.rc == 0 and r.launches, (line, r)
