"""How k_gemm_i8_batched reads and writes rows of any length (gemm_batched.hip):
a grid of more than one round of blocks, operands and results at odd addresses up
to the last byte of their buffers, results next to memory that must stay as it is;
and the pieces in which a tile leaves LDS (gemm_batched_out.h, built for the host)."""
import csv
import ctypes
import math
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "onnx-mlir_amd", "csrc")
DIRECT, TILE, ROWS = 0, 1, 2  # OutForm


@pytest.fixture(scope="module")
def out(tmp_path_factory):
    """What a launch and a block ask gemm_batched_out.h."""
    folder = tmp_path_factory.mktemp("out")
    (folder / "out.cpp").write_text("""
#include "gemm_batched_out.h"
using namespace om::gemm;
extern "C" {
int form(bool int32, int64_t M, int64_t N, uint64_t out, int64_t entries) {
  const int tiles_m = (int)((M + 63) / 64), tiles_n = (int)((N + 127) / 128);
  return out_form(int32, M, N, tiles_m, tiles_n, out, entries * tiles_m * tiles_n);
}
int first(int skew, int bytes) { return tile_pieces(skew, bytes).first; }
int last(int skew, int bytes) { return tile_pieces(skew, bytes).last; }
int end(int skew, int bytes, int tid) { return tile_end(tile_pieces(skew, bytes), tid); }
}
""")
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, "-o", str(folder / "out.so"), str(folder / "out.cpp")])
    lib = ctypes.CDLL(str(folder / "out.so"))
    lib.form.argtypes = [ctypes.c_bool, ctypes.c_int64, ctypes.c_int64, ctypes.c_uint64, ctypes.c_int64]
    return lib


def test_how_results_leave(out):
    """One by one up to 256 blocks, where rows are whole lines, where the first result
    does not start on a multiple of four, in tiles of few results and above 48 MB."""
    at = 1 << 40
    for N in (33, 63, 100, 127):
        assert out.form(True, 64, N, at, 257) == TILE and out.form(True, 64, N, at, 256) == DIRECT
        assert out.form(True, 65, N, at, 300) == (TILE if 65 * N * 4 >= 2 * 6144 else DIRECT)
        for off in range(1, 16):
            assert out.form(True, 64, N, at + off, 300) == (DIRECT if off % 4 else TILE), off
            assert out.form(False, 64, N, at + off, 300) == DIRECT
    assert out.form(True, 64, 64, at, 300) == out.form(True, 64, 160, at, 300) == DIRECT
    assert [out.form(True, 64, N, at, 300) for N in (132, 133, 134, 196)] == [ROWS, DIRECT, DIRECT, ROWS]
    assert all(out.form(True, 64, 132, at + off, 300) == DIRECT for off in range(1, 16)) and out.form(False, 64, 132, at, 300) == DIRECT
    assert [out.form(True, M, 48, at, 300) for M in (31, 32)] == [DIRECT, TILE]
    assert [out.form(True, M, 196, at, 300) for M in (15, 16)] == [DIRECT, ROWS]
    assert [out.form(True, 64, 100, at, n) for n in (48000000 // 25600, 48000000 // 25600 + 1)] == [TILE, DIRECT]


def test_the_way_out_is_the_faster_one_measured(out):
    """Up to 75 MB, where it does not depend on what the last-level cache holds."""
    over, never = [], []
    with open(os.path.join(os.path.dirname(os.path.dirname(CSRC)), "profiles", "batched_way_out_times.csv")) as f:
        for r in csv.DictReader(line for line in f if not line.startswith("#")):
            E, M, N, direct, lds = int(r["entries"]), int(r["M"]), int(r["N"]), float(r["direct"]), float(r["by_lds"])
            if E * M * N * 4 > 75e6:
                continue
            form = out.form(r["results"] == "i32", M, N, 1 << 40, E)
            over.append((direct if form == DIRECT else lds) / min(direct, lds))
            never.append(direct / min(direct, lds))
    assert len(over) > 700
    assert math.exp(np.mean(np.log(over))) < 1.01 < math.exp(np.mean(np.log(never))), (over, never)


@pytest.mark.parametrize("count", [1, 2, 3, 4, 5, 15, 16, 17, 31, 33, 64 * 7, 64 * 127, 64 * 100 + 1])
def test_a_tile_leaves_in_pieces_that_cover_it_once(out, count):
    """tile_out: aligned pieces of 16 bytes and single results at the two ends, from
    every address that out_form lets through."""
    size = count * 4
    for skew in range(16):
        if out.form(True, 64, 63, (1 << 40) + skew, 300) != TILE:
            continue
        written = [(o, 16) for t in range(256) for o in range(out.first(skew, size) + t * 16, out.last(skew, size), 256 * 16)]
        written += [(o, 4) for o in (out.end(skew, size, t) for t in range(256)) if o >= 0]
        covered = np.zeros(skew + size + 16, int)
        for o, n in written:
            covered[o:o + n] += 1
        assert (covered[skew:skew + size] == 1).all() and covered.sum() == size, skew
    assert 15 + 64 * 128 * 4 <= 64 * (128 * 4 + 32)  # the LDS it lies in


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


@pytest.mark.gpu
@pytest.mark.parametrize("count,M,K,N", [(300, 5, 16, 7), (260, 64, 63, 100), (130, 65, 32, 132)])
@pytest.mark.parametrize("off", [1, 2, 3])
def test_int32_results_that_start_between_words(rt, oracle, count, M, K, N, off):
    rng = np.random.default_rng(M + off)
    a, b = rng.integers(0, 256, (count, M, K), dtype=np.uint8), rng.integers(-128, 128, (count, K, N), dtype=np.int8)
    want = np.matmul(a.astype(np.int32), b.astype(np.int32))
    whole = rt.DeviceArray.from_numpy(np.full(want.nbytes + 64, 90, np.uint8))
    y = rt.DeviceArray.view_of(whole, 32 + off, (want.nbytes,))
    y.shape, y.dtype, y.size = want.shape, want.dtype, want.size
    rt.MatMulInteger(rt.DeviceArray.from_numpy(a), rt.DeviceArray.from_numpy(b), None, None, out=y)
    rt.synchronize()
    assert rt.last_gemm_kernel() == "k_gemm_i8_batched"
    got = whole.numpy()
    assert np.array_equal(got[32 + off:][:want.nbytes].view(np.int32).reshape(want.shape), want)
    assert (got[:32 + off] == 90).all() and (got[32 + off + want.nbytes:] == 90).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N,form", [(64, 63, 100, TILE), (40, 48, 62, TILE), (65, 33, 132, ROWS), (66, 130, 196, ROWS), (9, 65, 33, DIRECT)])
@pytest.mark.parametrize("alead,blead", [((10, 1, 3), (10, 9, 1)), ((270,), (270,)), ((1,), (270,))])
@pytest.mark.parametrize("adt,bdt", [(np.uint8, np.int8), (np.int8, np.uint8)])
def test_every_way_out_with_zero_points_of_every_row_and_column(rt, out, M, K, N, form, alead, blead, adt, bdt):
    """270 entries: in batch dimensions that do not merge (the general form of the
    arguments) and in one, each matrix of B with one of A or all with the same, int8
    and uint8 on either side."""
    rng = np.random.default_rng(M + K + N)
    i, j = np.iinfo(adt), np.iinfo(bdt)
    a, b = rng.integers(i.min, i.max + 1, alead + (M, K), dtype=adt), rng.integers(j.min, j.max + 1, blead + (K, N), dtype=bdt)
    az, bz = rng.integers(i.min, i.max + 1, alead + (M, 1), dtype=adt), rng.integers(j.min, j.max + 1, blead + (1, N), dtype=bdt)
    for azp, bzp in ((az, bz), (az.reshape(-1)[:1].reshape(()), bz), (None, None)):
        want = np.matmul(a.astype(np.int32) - (0 if azp is None else azp.astype(np.int32)), b.astype(np.int32) - (0 if bzp is None else bzp.astype(np.int32)))
        y = rt.DeviceArray(want.shape, np.int32)
        assert out.form(True, M, N, y.ptr, 270) == form
        rt.MatMulInteger(*(None if v is None else rt.DeviceArray.from_numpy(v) for v in (a, b, azp, bzp)), out=y)
        rt.synchronize()
        assert rt.last_gemm_kernel() == "k_gemm_i8_batched"
        assert np.array_equal(y.numpy(), want), (azp is None, bzp is None)
