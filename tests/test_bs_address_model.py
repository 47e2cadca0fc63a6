"""Host model of the memory accesses of the tile kernels in gemm_bs.hip beside
those of A (test_bs_line_model.py): weights, results at the edges and inside, parts
of K; of the copies to an aligned pitch (k_pad_rows) and the chunks that the
weight-streaming kernel reads at any address; and of the buffer pool's size
arithmetic (runtime.hip).  No GPU: the index arithmetic restated for the host,
lane by lane, and checked against the extents of the operands.

Step counts of every kind are among the shapes, 17 above all: an earlier form of
the streaming kernel ended a benchmark loop on 4096 x 1088 x 4096 with an illegal
access.  Its addresses were in bounds as well; what went wrong is in
test_loads_in_flight.py, which holds for the kernels of today that it cannot
happen, and the loop's waits are in test_bs_line_model.py."""
import os
import re

import numpy as np
import pytest

BK = 64
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = open(os.path.join(ROOT, "onnx-mlir_amd", "csrc", "gemm_bs.hip")).read()
LANE = np.arange(64)
L32, LH = LANE & 31, LANE >> 5


def round_up(a, b):
    return (a + b - 1) // b * b


# ---------------------------------------------------------------------------
# block -> tile (XCD interleave, then groups of 8 row tiles)
# ---------------------------------------------------------------------------
def tile_of(pid, nb, tiles_m, tiles_n):
    per = nb >> 3
    if per > 0 and pid < per * 8:
        pid = (pid & 7) * per + (pid >> 3)
    group_rows = 8
    in_group = group_rows * tiles_n
    group = pid // in_group
    first_m = group * group_rows
    gsize = min(tiles_m - first_m, group_rows)
    tm = first_m + (pid % in_group) % gsize
    tn = (pid % in_group) // gsize
    return tm, tn


@pytest.mark.parametrize("tiles_m,tiles_n", [(32, 16), (33, 16), (1, 1), (7, 3), (8, 43), (17, 5), (64, 1), (3, 100)])
def test_every_tile_is_computed_exactly_once(tiles_m, tiles_n):
    nb = tiles_m * tiles_n
    seen = {tile_of(p, nb, tiles_m, tiles_n) for p in range(nb)}
    assert len(seen) == nb
    assert all(0 <= tm < tiles_m and 0 <= tn < tiles_n for tm, tn in seen)


# ---------------------------------------------------------------------------
# weights
# ---------------------------------------------------------------------------
def buffer_reads(offset, scalar, size):
    """Which 16-byte loads the device makes: those whose lane offset (with the
    instruction's own) is below the descriptor's size minus the scalar offset,
    unsigned."""
    return offset < (size - scalar) % 2 ** 32


SHAPES = [(4096, 1024, 4096), (4096, 1088, 4096), (2048, 4096, 11008), (4100, 1088, 4000), (129, 192, 257), (65, 16, 33),
          (300, 784, 130), (64, 64, 1), (4095, 2048, 8190), (1500, 16, 5120), (90, 4176, 300)]


@pytest.mark.parametrize("TN", [1, 2])
@pytest.mark.parametrize("M,K,N", SHAPES)
@pytest.mark.parametrize("part_steps", [0, 4, 12])
def test_weights_are_read_where_they_lie_and_nowhere_else(TN, M, K, N, part_steps):
    """Every step that a block asks for, the four that its last trip and its
    prefetch run past the end among them; part_steps: K split into parts (0: not)."""
    KTs = round_up(K, BK) // BK
    bp_bytes = round_up(N, 256) * KTs * BK
    parts = -(-KTs // part_steps) if part_steps else 1
    for part in {0, parts - 1}:
        kfirst = part * part_steps
        KT = min(part_steps, KTs - kfirst) if part_steps else KTs
        asked = round_up(KT, 4) + 3
        for tn in {0, (N - 1) // (128 * TN)}:
            for wave in range(4):
                ncol0 = tn * 128 * TN + wave * 32 * TN
                base = ((ncol0 >> 5) * KTs + kfirst) * 2048
                size = (TN - 1) * KTs * 2048 + KT * 2048
                assert base + size <= bp_bytes
                for step in range(asked):
                    inside = step < KT
                    for half in range(2):
                        for j in range(TN):
                            lane = j * KTs * 2048 + LANE * 16 + half * 1024
                            scalar = step * 2048 if inside else 0
                            read = buffer_reads(lane, scalar, size if inside else 0)
                            assert read.all() == read.any() == inside
                            if inside:
                                at = base + lane + scalar
                                want = (((ncol0 >> 5) + j) * KTs + kfirst + step) * 2048 + half * 1024 + LANE * 16
                                assert (at == want).all() and at.max() + 16 <= bp_bytes


def test_the_half_step_is_not_in_the_scalar_offset():
    """An empty descriptor with a scalar offset of 1024 would be read through."""
    assert buffer_reads(LANE * 16, 1024, 0).all()
    load = re.search(r"auto load_b = .*?\n  \};", SOURCE, re.S).group(0)
    assert "offen offset:%4" in load and "bstep" in load and "* 1024" not in load.split("asm volatile")[0]


# ---------------------------------------------------------------------------
# results
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("TM,TN", [(4, 2), (2, 2), (2, 1)])
@pytest.mark.parametrize("M,N", [(4096, 4096), (4100, 4000), (129, 257), (65, 33), (64, 1), (1, 130), (128, 31), (200, 8190)])
@pytest.mark.parametrize("es", [1, 4])
def test_results_are_stored_once_and_inside(TM, TN, M, N, es):
    """Whole wave tiles by scalar row offsets, cut ones through a descriptor that
    ends with the tile's last row: the elements that the device does not drop are
    those of the matrix, each in its place."""
    BM, BN = 32 * TM, 128 * TN
    r = np.arange(16)
    row_of = 8 * (r >> 2) + (r & 3)  # + 4 * lh
    for tm in {0, (M - 1) // BM}:
        for tn in {0, (N - 1) // BN}:
            for wave in range(4):
                m0, n0 = tm * BM, tn * BN + wave * 32 * TN
                rows, cols = M - m0, N - n0
                base = (m0 * N + n0) * es
                loff = (4 * LH * N + L32) * es
                if rows <= 0 or cols <= 0:
                    continue
                full = rows >= 32 * TM and cols >= 32 * TN
                nr, nc = min(rows, 32 * TM), min(cols, 32 * TN)
                size = 0x7FFFFFFF if full else ((nr - 1) * N + nc) * es
                stored = []
                for i in range(TM):
                    for j in range(TN):
                        lane = np.where(j * 32 + L32 < cols, loff + j * 32 * es, 0x80000000)
                        for rr in row_of:
                            rowb = (i * 32 + rr) * N * es
                            at = lane + rowb
                            assert at.max() < 2 ** 32
                            keep = at < size if not full else np.ones(64, bool)
                            m, n = m0 + i * 32 + rr + 4 * LH, n0 + j * 32 + L32
                            assert (keep == ((m < M) & (n < N))).all()
                            assert (base + at[keep] == ((m * N + n) * es)[keep]).all()
                            stored.append(at[keep])
                stored = np.concatenate(stored)
                assert len(stored) == nr * nc == len(np.unique(stored))
                assert base + stored.max() + es <= M * N * es


# ---------------------------------------------------------------------------
# 16-byte chunks at any address
# ---------------------------------------------------------------------------
def chunk(a, M, K, row, k0, fill, length):
    """row_chunk (gemm_common.h) of the 16 bytes loaded for chunk k0 of `row`: read
    at their address, or moved back to end with A; the bytes that are not the
    row's replaced.  `length`: how many are."""
    at, last = row * K + k0, M * K - 16
    start = min(at, last)
    assert 0 <= start and start + 16 <= M * K
    v = int.from_bytes(a.reshape(-1)[start:start + 16].tobytes(), "little")
    back = at - start
    lo, hi = v & (2 ** 64 - 1), v >> 64
    shift = back * 8 if length > 0 else 0
    if shift >= 64:
        lo, hi = hi, 0
    s1 = shift & 63
    if s1:
        lo, hi = ((lo >> s1) | (hi << (64 - s1))) & (2 ** 64 - 1), hi >> s1
    mlo = 2 ** 64 - 1 if length >= 8 else (1 << (8 * length)) - 1
    mhi = 2 ** 64 - 1 if length >= 16 else ((1 << (8 * (length - 8))) - 1 if length > 8 else 0)
    f = int.from_bytes(bytes([fill]) * 8, "little")
    lo, hi = (lo & mlo) | (f & ~mlo & (2 ** 64 - 1)), (hi & mhi) | (f & ~mhi & (2 ** 64 - 1))
    return np.frombuffer((lo | hi << 64).to_bytes(16, "little"), np.uint8)


@pytest.mark.parametrize("M,K", [(65, 1), (70, 3), (129, 15), (66, 17), (200, 64), (65, 1019), (33, 4101), (1, 17), (16, 1), (7, 3),
                                 (2, 9), (5, 356)])
def test_padded_rows_hold_the_row_and_its_zero_point(M, K):
    rng = np.random.default_rng(M + K)
    a, zp = rng.integers(0, 256, (M, K), dtype=np.uint8), rng.integers(0, 256, M, dtype=np.uint8)
    Kp = round_up(K, 64)
    chunks = Kp // 16
    rows = range(M) if M * chunks < 2000 else [0, 1, M - 2, M - 1]
    for r in rows:  # thread r * chunks + c
        got = np.concatenate([chunk(a, M, K, r, c * 16, zp[r], max(0, min(16, K - c * 16))) for c in range(chunks)])
        assert np.array_equal(got, np.concatenate([a[r], np.full(Kp - K, zp[r], np.uint8)]))
    assert M * chunks * 16 == M * Kp  # what the runtime asks the pool for


# ---------------------------------------------------------------------------
# the pool
# ---------------------------------------------------------------------------
def test_pool_blocks_are_never_smaller_than_asked_for():
    """Ctx::take: the request rounded up to 256 bytes; an idle block serves it
    if it is the smallest one that is large enough and at most twice as large."""
    rng = np.random.default_rng(0)
    pool = []  # capacities of idle blocks
    for _ in range(2000):
        want = int(rng.integers(0, 1 << 24))
        need = round_up(max(want, 16) if want else 16, 256)
        fits = sorted(c for c in pool if c >= need)
        if fits and fits[0] <= 2 * need:
            cap = fits[0]
            pool.remove(cap)
        else:
            cap = need
        assert cap >= want and cap >= need
        if rng.integers(0, 2):
            pool.append(cap)
    for want in (4096 * 1088, 1088 * 4096, 4096 * 4096 * 4):
        assert round_up(want, 256) >= want
