"""Host model of k_gemm_i8_bs and k_gemm_i8_dma_bs, A copied in stages of two K
steps (onnx-mlir_amd/csrc/gemm_bs.hip): where their copies and operand reads go,
and whether its explicit waits cover what each step reads.  Index arithmetic
restated for the CPU (weights, results, parts of K: test_bs_address_model.py; the
registers that loads are still to write: test_loads_in_flight.py); and the kernels
themselves on the GPU, forced, at their edges."""
import numpy as np
import pytest

D, NST, ROW, BK = 4, 4, 128, 64
LANE = np.arange(64)
TILES = [(4, 2), (2, 2), (2, 1)]  # TM, TN


def slot_of(row, chunk):
    return row * ROW + ((chunk ^ ((row >> 1) & 7)) << 4)


@pytest.mark.parametrize("TM", [4, 2])
@pytest.mark.parametrize("M,K", [(128, 256), (1, 256), (300, 512), (2048, 11008), (129, 4096), (65, 16), (100, 784)])
def test_copies_are_in_bounds_and_lie_where_operands_are_read(TM, M, K):
    BM = 32 * TM
    CA = BM // 32
    pairs = np.arange(-(-K // 128))  # past the last one the descriptor is empty
    for m0 in {0, (M - 1) // BM * BM}:
        a_bytes = min(M - m0, BM) * K
        filled = np.zeros(BM * ROW, bool)
        for wave in range(4):
            for h in range(CA):
                r = (wave * CA + h) * 8 + (LANE >> 3)
                chunk = (LANE & 7) ^ ((r >> 1) & 7)
                rc = np.where(m0 + r < M, r, M - 1 - m0)
                at = pairs[:, None] * ROW + (rc * K + chunk * 16)[None]
                # a chunk lies wholly inside the tile's rows or the descriptor drops it
                assert at.min() >= 0 and ((at + 16 <= a_bytes) | (at >= a_bytes)).all()
                inside = pairs[:, None] * ROW + (chunk * 16)[None] < K
                assert (at[inside] + 16 <= a_bytes).all()
                dst = (wave * CA + h) * 1024 + LANE * 16
                assert (dst == slot_of(r, chunk)).all()
                filled[dst[:, None] + np.arange(16)] = True
        assert filled.all()
    l32, lh = LANE & 31, LANE >> 5
    ra = l32 * ROW + ((lh ^ ((l32 >> 1) & 7)) << 4)
    for h in range(4):
        for i in range(TM):
            at = (ra ^ (h << 5)) + i * 32 * ROW
            assert (at == slot_of(i * 32 + l32, h * 2 + lh)).all()
            # 16 lanes at a time over the 64 banks: no two in one place
            for g in range(4):
                assert len(set((at[g * 16:g * 16 + 16] % 256) // 16)) == 16


KTS = [1, 2, 3, 4, 5, 8, 12, 17, 18, 64, 172]


@pytest.mark.parametrize("TM,TN", TILES)
@pytest.mark.parametrize("KT", KTS)
def test_waits_cover_what_each_step_reads(TM, TN, KT):
    """One wave's vector memory operations in issue order, over the whole trips of
    four steps that the loop makes for KT of them."""
    CA, CB = TM, 2 * TN
    ops = []  # (kind, asked for, register set or stage), in issue order

    def copy(pair):
        ops.extend([("a", pair, pair % NST)] * CA)

    def weights(step):
        ops.extend([("b", step, step % D)] * CB)

    def landed(kind, what, where, young):
        at = [i for i, o in enumerate(ops) if o[0] == kind and o[2] == where]
        assert ops[at[-1]][1] == what and at[-1] < len(ops) - young, (kind, what, young)

    young = 2 * CB + CA
    copy(0)
    for u in range(D - 1):
        weights(u)
        if u == 0:
            copy(1)
    landed("a", 0, 0, 3 * CB + CA)
    for p in range(-(-KT // D) * D // 2):
        landed("b", 2 * p, 2 * p % D, young)
        copy(p + 2)
        weights(2 * p + 3)
        landed("b", 2 * p + 1, (2 * p + 1) % D, young)
        landed("a", p + 1, (p + 1) % NST, young)
        weights(2 * p + 4)


@pytest.mark.parametrize("KT", KTS)
def test_no_stage_is_overwritten_while_a_wave_may_read_it(KT):
    """Barriers, one at the start and one at the top of every odd step: between two
    of them a wave may be anywhere.  A copy may land as soon as the fastest wave
    asks for it, and a read may happen as late as the slowest one's next barrier
    (it waits for its reads before that)."""
    steps = -(-KT // D) * D
    passed = {s: 1 + (s + 1) // 2 for s in range(steps)}  # in step s
    reads, copies = [], [(0, 0), (0, 1)]  # (barriers passed, pair)
    reads.append((1, 0))  # first operands, behind the first barrier
    for s in range(steps):
        p = s // 2
        if s % 2 == 0:
            reads += [(passed[s], p), (passed[s], p)]
            copies.append((passed[s], p + NST - 2))
        else:
            reads += [(passed[s], p), (passed[s], p + 1)]
    for at_copy, pair in copies:
        for at_read, other in reads:
            if other % NST != pair % NST:
                continue
            if other < pair:  # the stage's earlier contents: read before a barrier that the copy is behind
                assert at_read < at_copy, (pair, other, at_copy, at_read)
            elif other == pair:  # its own: read behind a barrier that follows the copy and its wait
                assert at_read > at_copy or pair == 0, (pair, at_copy, at_read)


@pytest.mark.gpu
@pytest.mark.parametrize("tile,name", [("2", "k_gemm_i8_bs"), ("6", "k_gemm_i8_dma_bs (64x256"), ("7", "k_gemm_i8_dma_bs (64x128")])
@pytest.mark.parametrize("M,K,N", [(128, 256, 256), (127, 512, 255), (129, 768, 257), (300, 1280, 513), (1024, 512, 768),
                                   (65, 16, 33), (63, 64, 127), (190, 400, 129), (513, 832, 300), (66, 1136, 260)])
def test_streaming_kernels_at_their_edges(rt, oracle, monkeypatch, tile, name, M, K, N):
    """Rows and columns past the result, a K of one chunk up to several trips and
    any number of steps and chunks past them; row sums, per-row zero points, the
    three epilogues."""
    rng = np.random.default_rng(M + K + N)
    monkeypatch.setenv("OM_MI355X_GEMM_TILE", tile)

    def draw(dt, shape):
        i = np.iinfo(dt)
        return rng.integers(i.min, i.max + 1, shape, dtype=dt)

    for adt, bdt, per in ((np.uint8, np.int8, False), (np.uint8, np.uint8, False), (np.int8, np.uint8, True),
                          (np.int8, np.int8, True)):
        a, b = draw(adt, (M, K)), draw(bdt, (K, N))
        az, bz = draw(adt, (M,) if per else ()), draw(bdt, (N,) if per else ())
        want = oracle.matmul_integer(a, b, az, bz)
        assert np.array_equal(rt.MatMulInteger(a, b, az, bz), want)
        if K % 256 == 0 or tile != "2":
            assert name in rt.last_gemm_kernel(), rt.last_gemm_kernel()
        if not per:
            s = rng.uniform(1e-3, 1e-2, N).astype(np.float32)
            got = rt.MatMulIntegerDequant(a, b, az, bz, np.float32(0.01), s)
            assert np.array_equal(got, oracle.dequant_epilogue(want, np.float32(0.01), s))
        if adt == bdt:
            q = [np.float32(v) for v in (0.0173, 0.005, 0.37)]
            y = oracle.qlinear_matmul(a, q[0], az.reshape(-1)[:1], b, q[1], bz.reshape(-1)[:1], q[2], az.reshape(-1)[0], 0)
            assert np.array_equal(rt.QLinearMatMul(a, q[0], az.reshape(-1)[:1], b, q[1], bz.reshape(-1)[:1], q[2],
                                                   az.reshape(-1)[0], rt.WRAP), y)


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N", [(65, 2128, 65), (200, 3056, 129), (90, 4176, 300)])
def test_streaming_kernel_split_along_k(rt, oracle, M, K, N):
    """Parts of whole trips, the last one of fewer steps and ending inside one."""
    rng = np.random.default_rng(K)
    a, b = rng.integers(0, 256, (M, K), dtype=np.uint8), rng.integers(0, 256, (K, N), dtype=np.uint8)
    az, bz = np.uint8(131), rng.integers(0, 256, N, dtype=np.uint8)
    assert np.array_equal(rt.MatMulInteger(a, b, az, bz), oracle.matmul_integer(a, b, az, bz))
    kernel = rt.last_gemm_kernel()
    assert "dma_bs" in kernel and "split" in kernel and "ragged" in kernel, kernel


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N,offset", [(154, 1022, 258, 0), (443, 967, 419, 0), (900, 1019, 640, 0), (107, 2009, 620, 0),
                                          (660, 1020, 474, 0), (154, 1024, 258, 1), (70, 1007, 200, 3)])
def test_rows_copied_to_an_aligned_pitch(rt, oracle, M, K, N, offset):
    """Rows of an awkward length or start, copied in chunks of 16 bytes read at any
    address (`offset`: bytes in front of A) with tails of zero points."""
    rng = np.random.default_rng(M + K)
    for adt, bdt, per in ((np.uint8, np.int8, False), (np.int8, np.uint8, True), (np.uint8, np.uint8, False)):
        i, j = np.iinfo(adt), np.iinfo(bdt)
        a, b = rng.integers(i.min, i.max + 1, (M, K), dtype=adt), rng.integers(j.min, j.max + 1, (K, N), dtype=bdt)
        az, bz = rng.integers(i.min, i.max + 1, M, dtype=adt), rng.integers(j.min, j.max + 1, N, dtype=bdt)
        az, bz = (az, bz) if per else (az[:1], bz[:1])
        whole = rt.DeviceArray.from_numpy(np.concatenate([np.full(offset, 77, adt), a.reshape(-1)]))
        da = rt.DeviceArray.view_of(whole, offset, (M, K))
        got = rt.MatMulInteger(da, rt.DeviceArray.from_numpy(b), rt.DeviceArray.from_numpy(az), rt.DeviceArray.from_numpy(bz))
        rt.synchronize()
        if M * N > 300000:
            assert "any K" not in rt.last_gemm_kernel(), rt.last_gemm_kernel()
        assert np.array_equal(got.numpy(), oracle.matmul_integer(a, b, az, bz))
    x, s = rng.standard_normal((M, K), dtype=np.float32), rng.uniform(1e-3, 1e-2, N).astype(np.float32)
    q, qs, qz = oracle.dynamic_quantize_linear(x)
    got = rt.DynQuantMatMulDequant(x, b, bz, s)
    assert np.array_equal(got, oracle.dequant_epilogue(oracle.matmul_integer(q, b, qz, bz), qs, s))


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N,offset", [(1, 17, 5, 0), (16, 1, 40, 0), (7, 3, 33, 0), (7, 1, 20, 0), (2, 9, 64, 0), (4, 255, 100, 0),
                                          (5, 356, 70, 0), (13, 1001, 4200, 0), (16, 2049, 31, 0), (17, 130, 64, 0), (32, 1021, 100, 0),
                                          (24, 1537, 4200, 0), (33, 700, 50, 0), (48, 4097, 40, 0), (64, 333, 4200, 0),
                                          (50, 1031, 5000, 0), (6, 1024, 70, 5), (20, 256, 4200, 1), (60, 128, 30, 15), (3, 64, 9, 8)])
def test_few_rows_of_any_length(rt, oracle, M, K, N, offset):
    """The weight-streaming kernel reads rows where they lie: ends inside a chunk, a
    wave's slice past K, the last chunk of A, starts at any byte; and quantizes
    rows that float4 do not divide."""
    rng = np.random.default_rng(M + 7 * K)
    for adt, bdt, per in ((np.uint8, np.int8, False), (np.int8, np.uint8, True), (np.uint8, np.uint8, False), (np.int8, np.int8, True)):
        i, j = np.iinfo(adt), np.iinfo(bdt)
        a, b = rng.integers(i.min, i.max + 1, (M, K), dtype=adt), rng.integers(j.min, j.max + 1, (K, N), dtype=bdt)
        az, bz = rng.integers(i.min, i.max + 1, M, dtype=adt), rng.integers(j.min, j.max + 1, N, dtype=bdt)
        az, bz = (az, bz) if per else (az[:1], bz[:1])
        whole = rt.DeviceArray.from_numpy(np.concatenate([np.full(offset, 77, adt), a.reshape(-1)]))
        da = rt.DeviceArray.view_of(whole, offset, (M, K))
        got = rt.MatMulInteger(da, rt.DeviceArray.from_numpy(b), rt.DeviceArray.from_numpy(az), rt.DeviceArray.from_numpy(bz))
        rt.synchronize()
        assert "skinny" in rt.last_gemm_kernel() or M * K < 16, rt.last_gemm_kernel()
        want = oracle.matmul_integer(a, b, az, bz)
        assert np.array_equal(got.numpy(), want), (adt, bdt)
        x, s = rng.normal(0.3, 1, (M, K)).astype(np.float32), rng.uniform(1e-3, 1e-2, N).astype(np.float32)
        x[-1, -1] = 9.5  # the largest element is the very last one
        q, qs, qz = oracle.dynamic_quantize_linear(x)
        z = bz if bdt == np.uint8 else None
        got = rt.DynQuantMatMulDequant(rt.DeviceArray.from_numpy(x), rt.DeviceArray.from_numpy(b),
                                       None if z is None else rt.DeviceArray.from_numpy(z), rt.DeviceArray.from_numpy(s))
        rt.synchronize()
        assert "skinny" in rt.last_gemm_kernel()
        assert np.array_equal(got.numpy(), oracle.dequant_epilogue(oracle.matmul_integer(q, b, qz, z), qs, s)), (M, K, N)
        y = [np.float32(v) for v in (0.0173, 0.005, 0.37)]
        want = oracle.qlinear_matmul(a, y[0], az[:1], b, y[1], bz[:1], y[2], az[0], 1)
        assert np.array_equal(rt.QLinearMatMul(a, y[0], az[:1], b, y[1], bz[:1], y[2], az[0], rt.SATURATE), want)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", ["0", "1", "2", "3", "6", "7", ""])
@pytest.mark.parametrize("M,K,N", [(129, 256, 260), (256, 512, 256), (70, 1001, 33), (20, 640, 100), (3, 33, 70)])
def test_gelu_in_every_kernel(rt, oracle, monkeypatch, tile, M, K, N):
    """onnx.Gelu in the epilogue, whole and cut tiles, rows of whole and of partial
    lines, with and without row sums.  Tolerance: 4 units in the last place of erf
    (2^-22) times |0.5 x|, plus one rounding of the result."""
    if tile:
        monkeypatch.setenv("OM_MI355X_GEMM_TILE", tile)
    rng = np.random.default_rng(K)
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    ws, bias = rng.uniform(1e-5, 1e-3, N).astype(np.float32), rng.normal(0, 1, N).astype(np.float32)
    q, s, z = oracle.dynamic_quantize_linear(x)
    for bdt, bz in ((np.int8, None), (np.uint8, np.uint8(131))):
        j = np.iinfo(bdt)
        b = rng.integers(j.min, j.max + 1, (K, N), dtype=bdt)
        plain = oracle.dequant_epilogue(oracle.matmul_integer(q, b, z, bz), s, ws) + bias
        got = rt.DynQuantMatMulDequant(x, b, bz, ws, bias, activation=rt.ACTIVATION_GELU)
        want = oracle.gelu(plain).astype(np.float64)
        tol = np.abs(0.5 * plain.astype(np.float64)) * 2.0 ** -22 + np.abs(want) * 2.0 ** -23 + 1e-45
        assert (np.abs(got - want) <= tol).all(), rt.last_gemm_kernel()


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N,low", [
    (65, 257, 129, True), (127, 321, 300, True), (193, 130, 65, True), (1618, 653, 311, True),
    (300, 272, 200, True),
    (2637, 787, 995, None), (932, 1764, 746, None), (3694, 78, 4295, False)])
def test_any_k_in_tiles_of_64_rows(rt, oracle, M, K, N, low):
    """k_gemm_i8 takes 64 x 128 tiles where they are dealt out better: whole and cut
    tiles, last steps of every length, A at an odd address, with and without row
    sums.  Whole numbers: exact."""
    rng = np.random.default_rng(M + K)
    for bdt in (np.int8, np.uint8):
        i = np.iinfo(bdt)
        b = rng.integers(i.min, i.max + 1, (K, N), dtype=bdt)
        a = rng.integers(0, 256, (M, K), dtype=np.uint8)
        azp = np.uint8(77)
        bzp = np.uint8(131) if bdt == np.uint8 else None
        want = oracle.matmul_integer(a, b, azp, bzp)
        got = rt.MatMulInteger(a, b, azp, bzp)
        kernel = rt.last_gemm_kernel()
        if "any K" in kernel and "split" not in kernel:
            assert low is None or ("64x128" in kernel) == low, kernel
        assert np.array_equal(got, want), kernel
        whole = rt.DeviceArray.from_numpy(np.concatenate([np.full(3, 77, np.uint8), a.reshape(-1)]))
        got = rt.MatMulInteger(rt.DeviceArray.view_of(whole, 3, (M, K)), rt.DeviceArray.from_numpy(b),
                               rt.DeviceArray.from_numpy(np.array(azp)), bzp if bzp is None else rt.DeviceArray.from_numpy(np.array(bzp)))
        rt.synchronize()
        assert np.array_equal(got.numpy(), want), rt.last_gemm_kernel()
