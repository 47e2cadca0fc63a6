"""How k_gemm_i8_batched reads and writes rows of any length (gemm_batched.hip):
a grid of more than one round of blocks, operands and results at odd addresses up
to the last byte of their buffers, results next to memory that must stay as it is;
and the pieces in which a tile leaves LDS, restated for the CPU."""
import numpy as np
import pytest


@pytest.mark.parametrize("es", [1, 4])
@pytest.mark.parametrize("count", [1, 2, 3, 4, 5, 15, 16, 17, 31, 33, 64 * 7, 64 * 127, 64 * 100 + 1])
def test_a_tile_leaves_in_pieces_that_cover_it_once(es, count):
    """tile_out: aligned pieces of 16 bytes and single results at the two ends."""
    size, per = count * es, 16 // es
    for skew in range(0, 16, es):
        first, last = 16 if skew else 0, (skew + size) & ~15
        written = [(o, 16) for t in range(256) for o in range(first + t * 16, last, 256 * 16)]
        for t in range(2 * per):
            o = skew + t * es if t < per else max(first, last) + (t - per) * es
            if o < skew + size and (t >= per or o < first):
                written.append((o, es))
        covered = np.zeros(skew + size + 16, int)
        for o, n in written:
            covered[o:o + n] += 1
        assert (covered[skew:skew + size] == 1).all() and covered.sum() == size, skew
    assert 15 + 64 * 128 * es <= 64 * (128 * 4 + 32) // (4 // es)  # the LDS it lies in


@pytest.mark.gpu
@pytest.mark.parametrize("count,M,K,N", [(300, 5, 3, 7), (300, 8, 17, 33), (270, 33, 64, 63), (260, 65, 65, 1), (140, 70, 31, 127),
                                         (260, 64, 129, 64), (130, 3, 200, 132), (260, 1, 16, 260), (90, 66, 80, 196), (130, 9, 70, 131),
                                         (260, 64, 63, 100),
                                         (260, 20, 66, 1), (260, 20, 67, 2), (300, 7, 65, 3), (300, 3, 1, 6)])
@pytest.mark.parametrize("a_off,b_off,y_off", [(0, 0, 0), (1, 3, 1), (7, 2, 2), (16, 1, 3)])
def test_many_entries_at_any_address(rt, oracle, count, M, K, N, a_off, b_off, y_off):
    rng = np.random.default_rng(count + M * 100 + K * 10 + N)
    for adt, bdt in ((np.uint8, np.uint8), (np.int8, np.uint8)):
        i, j = np.iinfo(adt), np.iinfo(bdt)
        a = rng.integers(i.min, i.max + 1, (count, M, K), dtype=adt)
        b = rng.integers(j.min, j.max + 1, (count, K, N), dtype=bdt)
        az, bz, yz = adt(7), bdt(131), adt(9)
        acc = np.matmul(a.astype(np.int64) - int(az), b.astype(np.int64) - int(bz)).astype(np.int32)

        def put(values, off):
            whole = rt.DeviceArray.from_numpy(np.concatenate([np.full(off, 77, values.dtype), values.reshape(-1)]))
            return rt.DeviceArray.view_of(whole, off, values.shape)

        da, db = put(a, a_off), put(b, b_off)
        zeros = [rt.DeviceArray.from_numpy(np.array(z)) for z in (az, bz, yz)]
        s = np.float32(0.01)
        ds = rt.DeviceArray.from_numpy(np.array(s))
        dy = rt.DeviceArray.from_numpy(np.array(np.float32(0.8)))
        for dtype in (np.int32, adt):
            guard = np.full(count * M * N + 64, 90, dtype)
            whole = rt.DeviceArray.from_numpy(guard)
            y = rt.DeviceArray.view_of(whole, 32 + y_off, acc.shape)
            if dtype == np.int32:
                rt.MatMulInteger(da, db, zeros[0], zeros[1], out=y)
                want = acc
            else:
                rt.QLinearMatMul(da, ds, zeros[0], db, ds, zeros[1], dy, zeros[2], rt.SATURATE, out=y)
                f = acc.astype(np.float32) * ((s * s) / np.float32(0.8))
                want = np.clip(np.rint(f).astype(np.int64) + int(yz), i.min, i.max).astype(adt)
            rt.synchronize()
            assert rt.last_gemm_kernel() == "k_gemm_i8_batched"
            got = whole.numpy()
            assert np.array_equal(got[32 + y_off:32 + y_off + acc.size].reshape(acc.shape), want), (adt, dtype)
            assert (got[:32 + y_off] == 90).all() and (got[32 + y_off + acc.size:] == 90).all(), (adt, dtype)
