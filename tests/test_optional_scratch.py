"""Scratch that a product can do without is not asked for in a way that fails the
call."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_copied_rows_while_the_program_captures_a_graph(rt, oracle):
    """Rows of 1019 and 1020 bytes are copied to an aligned pitch first.  With a
    capture open on a stream of the program's own, an ordinary allocation is
    refused; before the rows were copied these products made none."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(5)
    cases = []
    for M, K, N in ((900, 1019, 640), (660, 1020, 474)):
        a, b = rng.integers(0, 256, (M, K), dtype=np.uint8), rng.integers(-127, 128, (K, N), dtype=np.int8)
        zps = np.array([131], np.uint8), np.array([7], np.int8)
        cases.append((a, b, zps, [rt.DeviceArray.from_numpy(v) for v in (a, b) + zps], rt.DeviceArray((M, N), np.int32)))

    def run(rows=None):
        for a, b, _, (da, db, az, bz), out in cases:
            if rows:
                da = rt.DeviceArray.view_of(da, 0, (rows, a.shape[1]))
                out = rt.DeviceArray.view_of(out, 0, (rows, b.shape[1]))
            rt.MatMulInteger(da, db, az, bz, out=out)
            assert rows or "any K" not in rt.last_gemm_kernel(), rt.last_gemm_kernel()

    run()  # (a kernel is loaded when it is first launched, which a capture refuses too)
    rt.synchronize()
    rt.clear_cache()  # the thread's pool of GPU memory
    for c in cases:
        rt.mark_constant(c[3][1])
    run(rows=2)  # packs the weights
    rt.synchronize()
    x = torch.ones(1024, device="cuda")
    torch.cuda.synchronize()
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=stream):
        y = x * 3.0
        run()
    rt.synchronize()
    for _ in range(3):
        x.add_(1.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, x * 3.0)
    for a, b, (az, bz), on_gpu, out in cases:
        assert np.array_equal(out.numpy(), oracle.matmul_integer(a, b, az, bz)), a.shape
        rt.unmark_constant(on_gpu[1])
