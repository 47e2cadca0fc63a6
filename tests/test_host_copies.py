"""Host tensors that are copied by kernels through page-locked memory."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 4095, 4096, 4097, 16383, 16385, 65535, 65537, 98303, 524288, 524289, 1048576, 1048577,
                               1300001, 2200003])
def test_sizes_around_chunks_pieces_and_limits(rt, n):
    """Results in chunks of 16 KiB up to 4 MiB, inputs in pieces of 256 KiB up to 2
    MiB, larger ones by the ways for them; lengths that are no whole vectors."""
    rng = np.random.default_rng(n)
    x = rng.integers(-128, 128, n, dtype=np.int8)
    s, z = np.float32(0.5), np.int8(3)
    guarded = np.full(n + 64, 7.0, np.float32)
    for _ in range(2):  # the second call finds the first one's bytes in the arena
        rt.DequantizeLinear(x, s, z, out=guarded[32:32 + n])
        assert np.array_equal(guarded[32:32 + n], (x.astype(np.float32) - 3.0) * 0.5)
        assert (guarded[:32] == 7.0).all() and (guarded[32 + n:] == 7.0).all()
        assert np.array_equal(rt.QuantizeLinear(guarded[32:32 + n], s, z), x)
        x = x[::-1].copy()


@pytest.mark.parametrize("M,K,N", [(1, 256, 16), (100, 768, 768), (300, 333, 500), (128, 768, 3072), (700, 512, 1500)])
def test_layers_and_several_results(rt, oracle, M, K, N):
    rng = np.random.default_rng(M)
    b, ws = rng.integers(-127, 128, (K, N), dtype=np.int8), rng.uniform(1e-3, 1e-2, N).astype(np.float32)
    for _ in range(2):
        x = rng.standard_normal((M, K), dtype=np.float32)
        q, s, z = oracle.dynamic_quantize_linear(x)
        gq, gs, gz = rt.DynamicQuantizeLinear(x)
        assert np.array_equal(gq, q) and np.float32(gs) == s and int(gz) == int(z)
        want = oracle.dequant_epilogue(oracle.matmul_integer(q, b, z, None), s, ws)
        assert np.array_equal(rt.DynQuantMatMulDequant(x, b, None, ws), want)
