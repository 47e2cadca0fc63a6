"""The last two K steps of k_gemm_i8, which stand apart from its loop: one step, two,
and odd and even counts of those in the loop, the last a whole one or not."""
import numpy as np
import pytest

import om_mi355x


@pytest.fixture(scope="module")
def rt():
    om_mi355x.load()
    return om_mi355x


def _check(rt, M, K, N, kernel):
    """A at an odd address, with and without row sums.  Whole numbers: exact."""
    rng = np.random.default_rng(M * K)
    for bdt in (np.int8, np.uint8):
        i = np.iinfo(bdt)
        a, b = rng.integers(0, 256, (M, K), dtype=np.uint8), rng.integers(i.min, i.max + 1, (K, N), dtype=bdt)
        az, bz = np.array(77, np.uint8), np.array(131, np.uint8) if bdt == np.uint8 else None
        whole = rt.DeviceArray.from_numpy(np.concatenate([np.full(1, 77, np.uint8), a.reshape(-1)]))
        got = rt.MatMulInteger(rt.DeviceArray.view_of(whole, 1, (M, K)), rt.DeviceArray.from_numpy(b),
                               rt.DeviceArray.from_numpy(az), None if bz is None else rt.DeviceArray.from_numpy(bz))
        rt.synchronize()
        assert rt.last_gemm_kernel() == "k_gemm_i8 (any K, any alignment" + kernel, rt.last_gemm_kernel()
        # (float64 holds sums of 2^16 products of 16 bits exactly)
        want = (a.astype(np.float64) - 77) @ (b.astype(np.float64) - (0 if bz is None else 131))
        assert np.array_equal(got.numpy(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("K", [17, 64, 65, 128, 130, 192, 200, 256, 257, 320, 321])
@pytest.mark.parametrize("M", [67, 129])
def test_counts_of_k_steps(rt, M, K):
    _check(rt, M, K, 70, "; 64x128 tiles)")


@pytest.mark.gpu
@pytest.mark.parametrize("K", [64, 65, 130, 190, 250, 300, 321, 400])
def test_counts_of_k_steps_in_tiles_of_128_rows(rt, K):
    _check(rt, 1366, K, 4429, ")")


@pytest.mark.gpu
@pytest.mark.parametrize("K", [1473, 1537, 1601, 1665, 2049, 1793])  # a last part of 4, 5, 1, 2, 3 and 4 steps
def test_counts_of_k_steps_of_the_last_part(rt, K):
    _check(rt, 67, K, 70, "; split along K)")
