"""Which kernel a product takes: the modelled times (gemm_kernels.hip) against the
times that were measured (profiles/*.csv), and the choice on the GPU."""
import csv
import ctypes
import math
import os
import re
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "onnx-mlir_amd", "csrc")
SOURCE = open(os.path.join(CSRC, "gemm_kernels.hip")).read()


def _coefficients(pattern):
    """The numbers of a TileCost: lone, step, rowsum, block4, block1, base, round."""
    block = re.search(pattern, SOURCE, re.S).group(1)
    return [[float(v) for v in re.findall(r"-?\d+(?:\.\d+)?", row)] for row in re.findall(r"\{k\w+,([^}]*)\}", block)]


def _us(cost, M, K, N, bytes_, rowsums):
    bm, bn, trip, lone, step, rowsum, block4, block1, base, round_ = cost
    blocks = -(-M // bm) * -(-N // bn)
    rounds = -(-blocks // 256)
    b = max(1.0, round_ * rounds + (1.0 - round_) * blocks / 256)
    steps = -(-K // (64 * trip)) * trip
    return base + steps * max(lone, step * rounds) * (1 + rowsum if rowsums else 1) + (block1 if bytes_ else block4) * b


def _table(name):
    with open(os.path.join(ROOT, "profiles", name)) as f:
        for r in csv.DictReader(line for line in f if not line.startswith("#")):
            yield r


def test_the_tile_with_the_least_modelled_time_is_the_fastest_measured():
    costs = _coefficients(r"kTileCosts\[\] = \{(.*?)\n\};")
    columns = ["dma_128x128", "dma_128x64", "bs_128x256", "bs_64x256", "bs_64x128"]
    assert [c[:2] for c in costs] == [[128, 128], [128, 64], [128, 256], [64, 256], [64, 128]]
    over = []
    for r in _table("tile_kernel_times.csv"):
        M, K, N = int(r["M"]), int(r["K"]), int(r["N"])
        can = [i for i, c in enumerate(columns) if r[c] and not (i == 2 and K % 256)]
        model = {i: _us(costs[i], M, K, N, r["results"] == "u8", r["rowsums"] == "1") for i in can}
        times = {i: float(r[columns[i]]) for i in can}
        over.append(times[min(can, key=model.get)] / min(times.values()))
    assert len(over) > 2000
    assert math.exp(np.mean(np.log(over))) < 1.006  # 1.0185 with the coefficients before
    assert sum(o > 1.1 for o in over) < 0.01 * len(over)


def test_tiles_of_awkward_rows():
    t128, = _coefficients(r"static constexpr TileCost t128 = (\{.*?\});")
    t64, = _coefficients(r"static constexpr TileCost t64 = (\{.*?\});")
    over = []
    for r in _table("awkward_row_times.csv"):
        sizes = int(r["M"]), int(r["K"]), int(r["N"]), r["results"] == "u8", r["rowsums"] == "1"
        small, large = float(r["any_64x128"]), float(r["any_128x128"])
        over.append((small if _us(t64, *sizes) < _us(t128, *sizes) else large) / min(small, large))
    assert len(over) > 500 and math.exp(np.mean(np.log(over))) < 1.012


@pytest.fixture(scope="module")
def plan(rt, tmp_path_factory):
    """(copied, parts, steps of a part) as the runtime library decides for rows of any
    length: what it asks before it launches a product."""
    folder = tmp_path_factory.mktemp("plan")
    (folder / "plan.cpp").write_text("""
#include "om_kernels.h"
extern "C" void plan(int64_t M, int64_t K, int64_t N, int bytes, int rowsums, int64_t *out) {
  om::GemmArgs g = {};
  g.A = (const void *)((uintptr_t)1 << 40); // (never read)
  g.a_unsigned = true;
  g.b_unsigned = rowsums;
  g.M = M, g.K = K, g.N = N;
  g.epi = bytes ? om::kEpiQ8 : om::kEpiI32;
  out[0] = om::gemm_padded_k(g) != 0;
  om::gemm_plan_split(g);
  out[1] = g.split.parts;
  out[2] = g.split.steps;
}
""")
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I", CSRC, "-I", os.path.join(ROOT, "include"),
                           "-I", "/opt/rocm/include", "-o", str(folder / "plan.so"), str(folder / "plan.cpp"), rt.LIB_PATH,
                           "-Wl,--allow-shlib-undefined", "-Wl,-rpath," + os.path.dirname(rt.LIB_PATH)])
    lib = ctypes.CDLL(str(folder / "plan.so"))
    lib.plan.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_int] * 2 + [ctypes.c_void_p]

    def ask(M, K, N, bytes_, rowsums):
        out = (ctypes.c_int64 * 3)()
        lib.plan(M, K, N, bytes_, rowsums, out)
        return bool(out[0]), out[1], out[2]
    return ask


def test_the_way_of_awkward_rows_is_the_fastest_measured(plan):
    """Copied first, split along K or in one piece of either tile: the library's choice
    between all of them, on their times."""
    t128, = _coefficients(r"static constexpr TileCost t128 = (\{.*?\});")
    t64, = _coefficients(r"static constexpr TileCost t64 = (\{.*?\});")
    over, longer = [], []
    for r in _table("awkward_row_times.csv"):
        sizes = int(r["M"]), int(r["K"]), int(r["N"]), r["results"] == "u8", r["rowsums"] == "1"
        steps = -(-sizes[1] // 64)
        # (parts of so many steps -> time; asked for n, there may be fewer)
        splits = {-(-steps // -(-steps // int(n[6:]))): float(t) for n, t in r.items() if n.startswith("split_") and t}
        ways = [float(r[n]) for n in ("any_64x128", "any_128x128", "rows_copied")] + list(splits.values())
        copied, parts, _ = plan(*sizes)
        if copied:
            taken = ways[2]
        elif parts > 1:  # (between the parts that were timed)
            taken = float(np.interp(math.log(parts), *zip(*((math.log(p), splits[p]) for p in sorted(splits)))))
        else:
            taken = ways[0] if _us(t64, *sizes) < _us(t128, *sizes) else ways[1]
        over.append(taken / min(ways))
        if min(ways) > 26:
            longer.append(over[-1])
    assert len(over) > 1200 and len(longer) > 150
    assert math.exp(np.mean(np.log(over))) < 1.008, math.exp(np.mean(np.log(over)))
    assert math.exp(np.mean(np.log(longer))) < 1.007, math.exp(np.mean(np.log(longer)))
    assert sum(o > 1.1 for o in over) < 0.02 * len(over)


@pytest.mark.parametrize("M,K,N,bytes_,rowsums", [(1178, 4084, 8832, False, False), (4095, 2749, 2584, False, True), (3882, 826, 10618, False, True),
                                                  (1905, 7689, 1664, True, False), (1092, 4017, 9663, False, False)])
def test_long_products_of_awkward_rows_are_copied_first(plan, M, K, N, bytes_, rowsums):
    assert plan(M, K, N, bytes_, rowsums)[0]


def _product(rt, oracle, M, K, N, bdt, rng):
    a, b = rng.integers(0, 256, (M, K), dtype=np.uint8), rng.integers(np.iinfo(bdt).min, np.iinfo(bdt).max + 1, (K, N), dtype=bdt)
    az, bz = np.array([120], np.uint8), np.array([100], np.uint8) if bdt == np.uint8 else None
    got = rt.MatMulInteger(a, b, az, bz)
    assert np.array_equal(got, oracle.matmul_integer(a, b, az, bz))
    return rt.last_gemm_kernel()


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N,bdt,kernel", [
    (667, 384, 9472, np.int8, "dma (128x128"),   # 8.5 us, in 128 x 64 tiles 9.5
    (1903, 304, 8576, np.uint8, "dma (128x128"),  # 17.3 / 19.9
    (2048, 768, 3072, np.uint8, "(64x128"),       # 10.5, in 128 x 256 tiles 12.4
])
def test_short_k_and_many_columns(rt, oracle, M, K, N, bdt, kernel):
    assert kernel in _product(rt, oracle, M, K, N, bdt, np.random.default_rng(M))


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N,offset", [(50, 1137, 9152, 0), (43, 9313, 400, 0), (54, 4604, 330, 2), (24, 5568, 300, 1),
                                          (33, 315, 8200, 3), (64, 1024, 8200, 1)])
def test_few_awkward_rows_that_are_copied_first(rt, oracle, M, K, N, offset):
    """Rows read often at odd addresses, copied to an aligned pitch: results with
    zero points per tensor and per row, with and without row sums."""
    rng = np.random.default_rng(M + K)
    for adt, bdt, per in ((np.uint8, np.int8, False), (np.int8, np.uint8, True)):
        i, j = np.iinfo(adt), np.iinfo(bdt)
        a, b = rng.integers(i.min, i.max + 1, (M, K), dtype=adt), rng.integers(j.min, j.max + 1, (K, N), dtype=bdt)
        az, bz = rng.integers(i.min, i.max + 1, M if per else 1, dtype=adt), rng.integers(j.min, j.max + 1, N if per else 1, dtype=bdt)
        whole = rt.DeviceArray.from_numpy(np.concatenate([np.full(offset, 77, adt), a.reshape(-1)]))
        da = rt.DeviceArray.view_of(whole, offset, (M, K))
        got = rt.MatMulInteger(da, *(rt.DeviceArray.from_numpy(v) for v in (b, az, bz)))
        rt.synchronize()
        assert np.array_equal(got.numpy(), oracle.matmul_integer(a, b, az, bz)), (adt, bdt)


def test_rows_are_copied_where_that_was_faster():
    """The rule of gemm_padded_k for up to 64 rows, on the times measured."""
    rule = re.search(r"odd \* M \* K > (\d+) && \(M > (\d+) \|\| odd == 4\);\s*return many \|\| \(M > 32 && N > (\d+)\)", SOURCE)
    most, few, columns = (int(v) for v in rule.groups())
    over = []
    for r in _table("few_row_times.csv"):
        M, K, N, offset = (int(r[k]) for k in ("M", "K", "N", "offset"))
        as_is, copied = float(r["as_they_lie"]), float(r["copied"])
        odd = sum((offset + i * K) % 4 != 0 for i in range(4))
        copy = (odd * M * K > most and (M > few or odd == 4)) or (M > 32 and N > columns)
        over.append((copied if copy else as_is) / min(as_is, copied))
    assert len(over) > 800 and math.exp(np.mean(np.log(over))) < 1.004  # 1.019 by K >= 4096 alone
