"""Parity of k_gemm_i8_flight -- the kernel for products that one round of
blocks covers (K = 512, 768 or 1024), and the dynamically quantized layer in
one launch -- with the CPU oracle, through the C-ABI.  Bit-exact, fp32
included (same sequence of correctly rounded operations)."""
import numpy as np
import pytest

import oracle_lib
from om_mi355x import workloads as wl

pytestmark = pytest.mark.gpu


def _rand_q(rng, dt, shape):
    info = np.iinfo(dt)
    return rng.integers(info.min, info.max + 1, shape, dtype=dt)


def bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


def same_f32(a, b):
    a, b = np.asarray(a, np.float32), np.asarray(b, np.float32)
    return a.shape == b.shape and bool(np.all((bits(a) == bits(b)) | (np.isnan(a) & np.isnan(b))))


def mm(oracle, A, B, a_zp, b_zp):
    """The oracle's MatMulInteger; large products through its OpenMP restatement
    of the reference's passes (pinned to the triple loop in test_oracle.py)."""
    big = A.shape[0] * A.shape[1] * B.shape[1] > 1 << 27
    return oracle.matmul_integer(A, B, a_zp, b_zp, passes=big)


SHAPES = [(65, 512, 100), (128, 768, 768), (200, 1024, 1000), (512, 1024, 4096), (1000, 768, 416),
          (2048, 768, 256), (97, 768, 33), (1000, 512, 1024), (256, 1024, 2048)]


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_one_round_kernel_all_operand_types_and_epilogues(rt, oracle, M, K, N):
    """Every pair of operand types, zero points absent / scalar / per row and per
    column, and the three epilogues (int32; f32 with per-column scale, bias and
    Relu; 8-bit requantize, wrapping and saturating) on shapes with ragged edges
    in both directions that the dispatch gives to k_gemm_i8_flight."""
    rng = np.random.default_rng(M * 7 + K + N)
    for adt, bdt in ((np.uint8, np.int8), (np.int8, np.uint8), (np.uint8, np.uint8), (np.int8, np.int8)):
        A, B = _rand_q(rng, adt, (M, K)), _rand_q(rng, bdt, (K, N))
        az, bz = _rand_q(rng, adt, (M,)), _rand_q(rng, bdt, (N,))
        for a_zp, b_zp in ((None, None), (az[:1], None), (az[:1], bz[:1]), (az, bz)):
            want = mm(oracle, A, B, a_zp, b_zp)
            got = rt.MatMulInteger(A, B, a_zp, b_zp)
            # (one zero point per row of A is left to the other kernels)
            assert ("flight" in rt.last_gemm_kernel()) == (a_zp is None or a_zp.size == 1), rt.last_gemm_kernel()
            assert np.array_equal(got, want), (adt, bdt, a_zp is not None, b_zp is not None)
        acc = mm(oracle, A, B, az[:1], bz[:1])
        a_s = np.float32(0.0173)
        bs = rng.uniform(1e-3, 1e-2, N).astype(np.float32)
        bias = rng.normal(0, 2, N).astype(np.float32)
        want = oracle.dequant_epilogue(acc, a_s, bs) + bias
        assert same_f32(rt.MatMulIntegerDequant(A, B, az[:1], bz[:1], a_s, bs, bias), want)
        assert same_f32(rt.MatMulIntegerDequant(A, B, az[:1], bz[:1], a_s, bs, bias, activation=1),
                        np.fmax(want, np.float32(0)))
        assert "flight" in rt.last_gemm_kernel()
        if adt == bdt:
            ys = np.float32(0.37)
            yz = _rand_q(rng, adt, ())
            for mode, omode in ((rt.WRAP, oracle_lib.WRAP), (rt.SATURATE, oracle_lib.SATURATE)):
                want = oracle.qlinear_matmul(A, a_s, az[:1], B, np.float32(0.005), bz[:1], ys, yz, omode)
                got = rt.QLinearMatMul(A, a_s, az[:1], B, np.float32(0.005), bz[:1], ys, yz, mode)
                assert "flight" in rt.last_gemm_kernel()
                assert np.array_equal(got, want), (adt, mode)


def test_one_round_kernel_is_forced_and_falls_through(rt, oracle, monkeypatch):
    """OM_MI355X_GEMM_TILE=5 names the kernel; a shape it does not take (K no
    multiple of 256, more blocks than one round) still computes, with another
    kernel."""
    monkeypatch.setenv("OM_MI355X_GEMM_TILE", "5")
    rng = np.random.default_rng(55)
    for (M, K, N), mine in (((300, 768, 500), True), ((300, 704, 500), False), ((8192, 768, 3072), False)):
        A, B = _rand_q(rng, np.uint8, (M, K)), _rand_q(rng, np.int8, (K, N))
        az = _rand_q(rng, np.uint8, ())
        assert np.array_equal(rt.MatMulInteger(A, B, az, None), mm(oracle, A, B, az, None)), (M, K, N)
        assert ("flight" in rt.last_gemm_kernel()) == mine, (M, K, N, rt.last_gemm_kernel())


@pytest.mark.parametrize("M,K,N", [(33, 768, 768), (128, 768, 768), (100, 512, 200), (512, 1024, 1024), (65, 1024, 97),
                                   (1024, 768, 768), (2048, 512, 100), (40, 768, 3072)])
def test_dynamically_quantized_layer_in_one_launch(rt, oracle, M, K, N):
    """DynamicQuantizeLinear -> MatMulInteger -> Cast -> Mul (-> Add -> Relu) as
    one launch of k_gemm_i8_flight: the blocks agree on minimum and maximum
    through the exchange slots, every block quantizes its own 32 rows.  Against
    the oracle's chain of the separate ops, bit for bit; host and GPU-resident
    operands; signed and unsigned weights, weight zero points; inputs whose
    minimum or maximum sits in the last (ragged) row block, NaN and infinities
    among the activations."""
    rng = np.random.default_rng(M + K * 3 + N)
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    x[M - 1, K - 1] = 7.5            # the maximum in the last row
    x[0, 0] = -6.25
    for bdt in (np.int8, np.uint8):
        W = _rand_q(rng, bdt, (K, N))
        ws = rng.uniform(1e-3, 1e-2, N).astype(np.float32)
        bias = rng.normal(0, 1, N).astype(np.float32)
        bz = _rand_q(rng, bdt, (N,))
        aq, a_s, a_zp = oracle.dynamic_quantize_linear(x)
        for b_zp in (None, bz[:1], bz):
            acc = mm(oracle, aq, W, a_zp, b_zp)
            want = oracle.dequant_epilogue(acc, a_s, ws)
            got = rt.DynQuantMatMulDequant(x, W, b_zp, ws)
            assert "flight (rows quantized" in rt.last_gemm_kernel(), rt.last_gemm_kernel()
            assert same_f32(got, want), (bdt, b_zp is not None)
        wantb = np.fmax(oracle.dequant_epilogue(mm(oracle, aq, W, a_zp, None), a_s, ws[:1]) + bias,
                        np.float32(0))
        assert same_f32(rt.DynQuantMatMulDequant(x, W, None, ws[:1], bias, activation=1), wantb)
    # GPU-resident operands, called repeatedly (the launch number in the slots moves on)
    dX, dW, dS = rt.DeviceArray.from_numpy(x), rt.DeviceArray.from_numpy(W), rt.DeviceArray.from_numpy(ws)
    dY = rt.DeviceArray((M, N), np.float32)
    rt.mark_constant(dW)
    acc = mm(oracle, aq, W, a_zp, None)
    want = oracle.dequant_epilogue(acc, a_s, ws)
    for _ in range(5):
        rt.DynQuantMatMulDequant(dX, dW, None, dS, out=dY)
    rt.synchronize()
    assert same_f32(dY.numpy(), want)
    rt.unmark_constant(dW)
    for d in (dX, dW, dS, dY):
        d.free()
    # special values: NaN is ignored by the minimum / maximum and quantizes to
    # the lower bound, infinities saturate (and make the scale infinite)
    x2 = x.copy()
    x2[3, 5] = np.nan
    aq, a_s, a_zp = oracle.dynamic_quantize_linear(x2)
    W = _rand_q(rng, np.int8, (K, N))
    want = oracle.dequant_epilogue(mm(oracle, aq, W, a_zp, None), a_s, ws)
    assert same_f32(rt.DynQuantMatMulDequant(x2, W, None, ws), want)
    x2[M // 2, 7] = np.inf
    aq, a_s, a_zp = oracle.dynamic_quantize_linear(x2)
    want = oracle.dequant_epilogue(mm(oracle, aq, W, a_zp, None), a_s, ws)
    assert same_f32(rt.DynQuantMatMulDequant(x2, W, None, ws), want)


def test_config1_is_one_launch(rt, oracle):
    c = wl.config1()
    aq, a_s, a_zp = oracle.dynamic_quantize_linear(c["A"])
    want = oracle.dequant_epilogue(oracle.matmul_integer(aq, c["B"], a_zp, c["b_zp"]), a_s, c["b_scale"])
    assert same_f32(rt.DynQuantMatMulDequant(c["A"], c["B"], c["b_zp"], c["b_scale"]), want)
    assert rt.last_gemm_kernel() == "k_gemm_i8_flight (rows quantized in the kernel)"


@pytest.mark.parametrize("mode", [0, 1])
def test_fused_layer_takes_an_activation_that_is_not_16_byte_aligned(rt, oracle, mode):
    """A GPU-resident activation that starts 4 bytes into its buffer (a view):
    the one-launch kernels want 16-byte rows, so the layer runs as
    DynamicQuantizeLinear + GEMM, whose quantize pass then stores the rows minus
    128 with a kernel that takes any alignment -- also when the quotient is
    computed as x * (1 / scale) (mode 1), where this used to be refused."""
    M, K, N = 72, 768, 256
    rng = np.random.default_rng(72 + mode)
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    W = _rand_q(rng, np.int8, (K, N))
    ws = rng.uniform(1e-3, 1e-2, N).astype(np.float32)
    buf = rt.DeviceArray.from_numpy(np.concatenate([np.zeros(1, np.float32), x.ravel()]))
    dx = rt.DeviceArray.__new__(rt.DeviceArray)
    dx.shape, dx.dtype, dx.ptr, dx.owner = (M, K), np.dtype(np.float32), buf.ptr + 4, buf
    aq, a_s, a_zp = oracle.dynamic_quantize_linear_mode(x, mode)
    want = oracle.dequant_epilogue(mm(oracle, aq, W, a_zp, None), a_s, ws)
    rt.set_quant_mode(mode)  # (what a model compiled with that option emits in front of each op)
    try:
        got = rt.DynQuantMatMulDequant(dx, W, None, ws)
    finally:
        rt.set_quant_mode(0)
    got = got.numpy() if hasattr(got, "numpy") else got
    assert "flight (rows quantized" not in rt.last_gemm_kernel()
    assert same_f32(got, want)
    buf.free()


def test_qlinear_matmul_with_a_scale_per_column(rt, oracle):
    """b_scale as one value per column of B (what a QDQ model with per-channel
    weights recomposes to).  PARITY UNPINNED against the reference, whose
    lowering refuses this form (QLinearMatMul.cpp:53-68): the expected values
    are its expression (:127-138) with column j's scale -- f32(acc) * ((a_scale
    * b_scale[j]) / y_scale), roundEven, + y_zp, narrowed -- over the oracle's
    exact int32 product, restated here in numpy; with all columns' scales equal
    that restatement is checked against the oracle's own QLinearMatMul first."""
    rng = np.random.default_rng(4242)

    def expect(A, a_s, az, B, bs, bz, y_s, yz, saturate):
        acc = mm(oracle, A, B, az, bz)
        s = (np.float32(a_s) * bs.astype(np.float32)) / np.float32(y_s)
        q = np.rint(acc.astype(np.float32) * s[None, :]).astype(np.int64) + int(yz)
        info = np.iinfo(yz.dtype)
        if saturate:
            return np.clip(q, info.min, info.max).astype(yz.dtype)
        return (q & 0xFF).astype(np.uint8).view(yz.dtype) if yz.dtype == np.int8 else (q & 0xFF).astype(np.uint8)

    for (M, K, N), adt in (((200, 1024, 1000), np.uint8), ((300, 768, 384), np.int8), ((48, 200, 130), np.uint8),
                            ((1024, 768, 3072), np.uint8)):
        A, B = _rand_q(rng, adt, (M, K)), _rand_q(rng, np.int8, (K, N))
        az, yz = _rand_q(rng, adt, ()), _rand_q(rng, adt, ())
        bz = _rand_q(rng, np.int8, (N,)) if M != 1024 else np.zeros(N, np.int8)
        a_s, y_s = np.float32(0.0173), np.float32(0.11)
        same = np.full(N, 0.004, np.float32)
        for sat, omode, mode in ((False, oracle_lib.WRAP, rt.WRAP), (True, oracle_lib.SATURATE, rt.SATURATE)):
            assert np.array_equal(expect(A, a_s, az, B, same, bz, y_s, yz, sat),
                                  oracle.qlinear_matmul(A, a_s, az, B, same[0], bz, y_s, yz, omode))
            bs = rng.uniform(1e-3, 8e-3, N).astype(np.float32)
            got = rt.QLinearMatMul(A, a_s, az, B, bs, bz, y_s, yz, mode)
            assert np.array_equal(got, expect(A, a_s, az, B, bs, bz, y_s, yz, sat)), (M, K, N, sat, rt.last_gemm_kernel())


def _limits(a):
    a = np.asarray(a, np.float32)
    return np.array([np.fmin.reduce(a, axis=None), np.fmax.reduce(a, axis=None)], np.float32)


@pytest.mark.parametrize("M,K,N,N2", [(128, 768, 3072, 768), (4096, 768, 3072, 768), (16, 4096, 1024, 512),
                                      # ragged rows and a last column tile past N in the weights-in-registers kernel
                                      (2945, 768, 3040, 416),
                                      (33, 200, 130, 70), (300, 768, 1000, 416), (2, 64, 8, 5),
                                      # second layer quantized inside its kernel: one round of blocks; every block for itself
                                      (128, 768, 1024, 768), (200, 512, 768, 1000), (8, 1024, 2048, 512), (16, 512, 2048, 11008)])
def test_chain_of_layers_hands_the_limits_on(rt, oracle, M, K, N, N2):
    """om_mi355x_DynQuantMatMulDequantLimits: y_limits of a layer is minimum and
    maximum of its result (NaN ignored), bit for bit what numpy finds in it,
    whatever kernel produced y (in its epilogue, or a pass over y behind it) and
    with bias, Relu or Gelu applied; a second layer given them as x_limits
    returns exactly what it returns without them, and what the oracle's chain of
    the separate ops gives.  Host and GPU-resident tensors."""
    rng = np.random.default_rng(M + N)
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    W1, W2 = _rand_q(rng, np.int8, (K, N)), _rand_q(rng, np.int8, (N, N2))
    s1 = rng.uniform(1e-3, 1e-2, N).astype(np.float32)
    s2 = rng.uniform(1e-3, 1e-2, N2).astype(np.float32)
    bias = rng.normal(0, 1, N).astype(np.float32)
    for act in (0, 1, 2):
        h_plain = rt.DynQuantMatMulDequant(x, W1, None, s1, bias, activation=act)
        h, hl = rt.DynQuantMatMulDequantLimits(x, W1, None, s1, bias, activation=act)
        assert same_f32(h, h_plain), (act, rt.last_gemm_kernel())
        assert same_f32(hl, _limits(h)), (act, hl, _limits(h), rt.last_gemm_kernel())
        y_plain = rt.DynQuantMatMulDequant(h, W2, None, s2)
        kernel = rt.last_gemm_kernel()
        y, yl = rt.DynQuantMatMulDequantLimits(h, W2, None, s2, x_limits=hl)
        assert rt.last_gemm_kernel() == kernel  # (known limits do not change the kernel)
        assert same_f32(y, y_plain), (act, kernel)
        assert same_f32(yl, _limits(y))
        if act != 2:  # (the oracle's Gelu differs from the kernel's in the last bits)
            aq, a_s, a_zp = oracle.dynamic_quantize_linear(h)
            assert same_f32(y, oracle.dequant_epilogue(mm(oracle, aq, W2, a_zp, None), a_s, s2))
    # GPU-resident, the limits never leave the GPU
    dx, dW1, dW2, ds1, ds2 = (rt.DeviceArray.from_numpy(v) for v in (x, W1, W2, s1, s2))
    dh, dhl = rt.DeviceArray((M, N), np.float32), rt.DeviceArray((2,), np.float32)
    dy = rt.DeviceArray((M, N2), np.float32)
    for _ in range(3):
        rt.DynQuantMatMulDequantLimits(dx, dW1, None, ds1, None, out=dh, activation=1, y_limits=dhl)
        rt.DynQuantMatMulDequantLimits(dh, dW2, None, ds2, None, out=dy, x_limits=dhl, want_limits=False)
    rt.synchronize()
    h = rt.DynQuantMatMulDequant(x, W1, None, s1, None, activation=1)
    assert same_f32(dh.numpy(), h) and same_f32(dhl.numpy(), _limits(h))
    assert same_f32(dy.numpy(), rt.DynQuantMatMulDequant(h, W2, None, s2))
    for d in (dx, dW1, dW2, ds1, ds2, dh, dhl, dy):
        d.free()


def test_limits_with_nan_infinities_and_the_other_quotient(rt, oracle):
    """NaN in the result is ignored by the limits (as the reductions of
    DynamicQuantizeLinear ignore it), infinities are not; limits handed to a
    layer under SetQuantMode(1) and (2) give what that mode gives without them;
    limits of the wrong size are refused."""
    rng = np.random.default_rng(99)
    M, K, N = 70, 320, 96
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    W = _rand_q(rng, np.int8, (K, N))
    s = rng.uniform(1e-3, 1e-2, N).astype(np.float32)
    bias = rng.normal(0, 1, N).astype(np.float32)
    bias[5], bias[9] = np.nan, np.inf
    h, hl = rt.DynQuantMatMulDequantLimits(x, W, None, s, bias)
    assert np.isnan(h[:, 5]).all() and same_f32(hl, _limits(h)) and hl[1] == np.inf
    bias[9] = 1.0
    h, hl = rt.DynQuantMatMulDequantLimits(x, W, None, s, bias)
    assert np.isfinite(hl).all() and same_f32(hl, _limits(h))
    W2 = _rand_q(rng, np.int8, (N, 40))
    s2 = rng.uniform(1e-3, 1e-2, 40).astype(np.float32)
    h = np.nan_to_num(h, nan=0.25)
    hl = _limits(h)
    try:
        for mode in (1, 2, 3):
            rt.set_quant_mode(mode)
            want = rt.DynQuantMatMulDequant(h, W2, None, s2)
            got, _ = rt.DynQuantMatMulDequantLimits(h, W2, None, s2, x_limits=hl, want_limits=False)
            assert same_f32(got, want), mode
            aq, a_s, a_zp = oracle.dynamic_quantize_linear_mode(h, mode)
            assert same_f32(got, oracle.dequant_epilogue(mm(oracle, aq, W2, a_zp, None), a_s, s2)), mode
    finally:
        rt.set_quant_mode(0)
    with pytest.raises(rt.RuntimeError_, match="limits"):
        rt.DynQuantMatMulDequantLimits(h, W2, None, s2, x_limits=np.zeros(3, np.float32))


@pytest.mark.parametrize("M,K,N", [(1, 16, 4), (5, 1, 9), (63, 15, 63), (64, 64, 64), (65, 65, 65), (64, 16, 128),
                                   (66, 48, 68), (130, 129, 127), (33, 200, 129), (128, 64, 132), (200, 320, 256)])
@pytest.mark.parametrize("adt,bdt", [(np.uint8, np.uint8), (np.int8, np.int8), (np.uint8, np.int8)])
def test_batched_kernel_edges(rt, oracle, M, K, N, adt, bdt):
    """k_gemm_i8_batched at the edges of its 64-row and 64- / 128-column tiles,
    one to five K steps, aligned and unaligned rows, zero points of every form,
    int32 and requantized results, and batch dimensions that broadcast against
    each other on either side."""
    rng = np.random.default_rng(M * 1000 + K * 10 + N)

    def rand(dt, shape):
        i = np.iinfo(dt)
        return rng.integers(i.min, i.max + 1, shape).astype(dt)

    for alead, blead in (((2, 3), (2, 3)), ((2, 1), (3,)), ((1,), (4,)), ((2, 1, 3), (2, 2, 1))):
        A, B = rand(adt, alead + (M, K)), rand(bdt, blead + (K, N))
        forms = ((rand(adt, ()), rand(bdt, ())), (None, None), (rand(adt, alead + (M, 1)), rand(bdt, blead + (1, N))))
        for az, bz in forms:
            got = rt.MatMulInteger(A, B, az, bz)
            a64 = A.astype(np.int64) - (0 if az is None else az.astype(np.int64))
            b64 = B.astype(np.int64) - (0 if bz is None else bz.astype(np.int64))
            assert np.array_equal(got, np.matmul(a64, b64)), (alead, blead, az is None)
        if A.size >= 16:  # (an A below one 16-byte load goes matrix by matrix)
            assert rt.last_gemm_kernel() == "k_gemm_i8_batched"
    s, ydt = np.float32(0.01), adt
    az, bz, yz = rand(adt, ()), rand(bdt, ()), rand(ydt, ())
    A, B = rand(adt, (3, M, K)), rand(bdt, (3, K, N))
    for mode in (rt.WRAP, rt.SATURATE):
        got = rt.QLinearMatMul(A, s, az, B, s, bz, np.float32(0.5), yz, mode)
        want = oracle.qlinear_matmul(A, s, az, B, s, bz, np.float32(0.5), yz, mode)
        assert np.array_equal(got, want)


@pytest.mark.parametrize("M", [1, 4, 5, 16, 17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("K,N", [(16, 40), (1008, 4096 + 33), (2064, 4097)])
def test_few_rows_tile_widths(rt, oracle, M, K, N):
    """The weight-streaming kernel on both sides of its row-tile edges and of the
    column counts from which a block takes two column tiles (K <= 1024, or rows
    it quantizes itself) or one of 32 columns (more than 32 rows): unsigned
    weights with a zero point per column (row sums of A, whose chunks past K are
    corrected for), and the fused layer, which quantizes up to 32 Ki elements in
    the kernel."""
    rng = np.random.default_rng(M * 7 + N)
    A, B = rng.integers(0, 256, (M, K)).astype(np.uint8), rng.integers(0, 256, (K, N)).astype(np.uint8)
    az, bz = np.uint8(131), rng.integers(0, 256, (N,)).astype(np.uint8)
    got = rt.MatMulInteger(A, B, az, bz)
    assert "skinny" in rt.last_gemm_kernel()
    assert np.array_equal(got, oracle.matmul_integer(A, B, az, bz))
    x = rng.standard_normal((M, K), dtype=np.float32)
    ws = rng.uniform(1e-3, 1e-2, N).astype(np.float32)
    q, s, z = oracle.dynamic_quantize_linear(x)
    want = oracle.dequant_epilogue(oracle.matmul_integer(q, B, z, bz), s, ws)
    got = rt.DynQuantMatMulDequant(x, B, bz, ws)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("per_thread", [2, 8, 16, 32, 56])
@pytest.mark.parametrize("extra", [-1, 0, 1, 7])
def test_dynamic_quantize_register_edges(rt, oracle, per_thread, extra):
    """DynamicQuantizeLinear around the tensor sizes where one launch keeps
    another number of float4 per thread (512 threads on each of the CUs), and
    beyond the largest, where the elements in front of the kept ones are reduced
    first and quantized by a second launch; the extremes lie at the first
    element, in the middle and at the last one."""
    n = rt.device_info()["cus"] * 512 * 4 * per_thread + extra
    rng = np.random.default_rng(per_thread)
    x = rng.standard_normal(n, dtype=np.float32)
    for at in (0, n // 2, n - 1):
        x[at], x[(at + 1) % n] = 11.0 + at % 3, -9.0
        wy, ws, wz = oracle.dynamic_quantize_linear(x)
        dy, ds, dz = rt.DynamicQuantizeLinear(rt.DeviceArray.from_numpy(x))
        rt.synchronize()
        assert ds.numpy().view(np.uint32) == np.float32(ws).view(np.uint32) and int(dz.numpy()) == int(wz)
        assert np.array_equal(dy.numpy(), wy)
        x[at] = x[(at + 1) % n] = 0.5


@pytest.mark.parametrize("K", [16, 48, 80, 784, 1008, 17, 63, 65, 127, 777])
def test_products_whose_rows_end_inside_a_k_step(rt, oracle, K):
    """K no multiple of 64: the last K step of k_gemm_i8_dma (K % 16 == 0) and
    of k_gemm_i8 (any K) covers chunks that are partly or wholly past the row,
    which must count neither in the products nor in the row sums; rows and
    columns past the edge of the result are dropped by its store descriptor.
    All operand types, zero points per tensor and per row / column, the three
    epilogues, results next to memory that must stay as it is."""
    rng = np.random.default_rng(K)
    for M, N in ((65, 33), (129, 100), (300, 1001)):
        for adt, bdt in ((np.uint8, np.int8), (np.int8, np.uint8), (np.uint8, np.uint8), (np.int8, np.int8)):
            A, B = _rand_q(rng, adt, (M, K)), _rand_q(rng, bdt, (K, N))
            az, bz = _rand_q(rng, adt, (M,)), _rand_q(rng, bdt, (N,))
            for a_zp, b_zp in ((None, None), (az[:1], bz), (az, bz[:1])):
                assert np.array_equal(rt.MatMulInteger(A, B, a_zp, b_zp), mm(oracle, A, B, a_zp, b_zp)), (M, N, adt, bdt)
            assert ("dma" in rt.last_gemm_kernel()) == (K % 16 == 0), rt.last_gemm_kernel()
            if adt == bdt:
                s = [np.float32(v) for v in (0.0173, 0.005, 0.37)]
                want = oracle.qlinear_matmul(A, s[0], az[:1], B, s[1], bz[:1], s[2], az[1], oracle_lib.WRAP)
                assert np.array_equal(rt.QLinearMatMul(A, s[0], az[:1], B, s[1], bz[:1], s[2], az[1], rt.WRAP), want)
        x = rng.normal(0, 1, (M, K)).astype(np.float32)
        ws, bias = rng.uniform(1e-3, 1e-2, N).astype(np.float32), rng.normal(0, 1, N).astype(np.float32)
        aq, a_s, a_zp = oracle.dynamic_quantize_linear(x)
        want = oracle.dequant_epilogue(mm(oracle, aq, B, a_zp, bz), a_s, ws) + bias
        assert same_f32(rt.DynQuantMatMulDequant(x, B, bz, ws, bias), want)
        # the result between two guards in one buffer
        guard = np.full(2 * 512 + M * N, 0x5A5A5A5A, np.int32)
        whole, dA, dB = (rt.DeviceArray.from_numpy(v) for v in (guard, A, B))
        rt.MatMulInteger(dA, dB, None, None, out=rt.DeviceArray.view_of(whole, 512, (M, N)))
        rt.synchronize()
        got = whole.numpy()
        assert np.array_equal(got[512:-512].reshape(M, N), mm(oracle, A, B, None, None))
        assert np.all(got[:512] == 0x5A5A5A5A) and np.all(got[-512:] == 0x5A5A5A5A)


@pytest.mark.parametrize("M,K,N", [(65, 2112, 65), (70, 2048, 33), (129, 4096, 258), (130, 2064, 257), (300, 4112, 130),
                                   (65, 1537, 66), (129, 2001, 129), (257, 4097, 33)])
def test_products_split_along_k(rt, oracle, monkeypatch, M, K, N):
    """Few tiles and many K steps: parts of K multiplied by blocks of their own
    and added up by k_sum_parts.  K of whole steps, of whole 16-byte chunks and
    odd, a last part shorter than the others, results whose length is no
    multiple of four and one that does not start on a 16-byte boundary; all
    operand types, zero points per tensor and per row / column (row sums of each
    part; whole-K terms once), the three epilogues, bias and activations, the
    latter against the same product in one piece."""
    rng = np.random.default_rng(K)
    for adt, bdt in ((np.uint8, np.int8), (np.int8, np.uint8), (np.uint8, np.uint8), (np.int8, np.int8)):
        A, B = _rand_q(rng, adt, (M, K)), _rand_q(rng, bdt, (K, N))
        az, bz = _rand_q(rng, adt, (M,)), _rand_q(rng, bdt, (N,))
        for a_zp, b_zp in ((None, None), (az[:1], bz), (az, bz[:1])):
            assert np.array_equal(rt.MatMulInteger(A, B, a_zp, b_zp), mm(oracle, A, B, a_zp, b_zp)), (adt, bdt)
            assert "split" in rt.last_gemm_kernel(), rt.last_gemm_kernel()
        if adt == bdt:
            s = [np.float32(v) for v in (0.0173, 0.005, 2.37)]
            for mode, rt_mode in ((oracle_lib.WRAP, rt.WRAP), (oracle_lib.SATURATE, rt.SATURATE)):
                want = oracle.qlinear_matmul(A, s[0], az[:1], B, s[1], bz[:1], s[2], az[1], mode)
                assert np.array_equal(rt.QLinearMatMul(A, s[0], az[:1], B, s[1], bz[:1], s[2], az[1], rt_mode), want)
                assert "split" in rt.last_gemm_kernel()
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    ws, bias = rng.uniform(1e-3, 1e-2, N).astype(np.float32), rng.normal(0, 1, N).astype(np.float32)
    aq, a_s, a_zp = oracle.dynamic_quantize_linear(x)
    plain = oracle.dequant_epilogue(mm(oracle, aq, B, a_zp, bz), a_s, ws)
    assert same_f32(rt.DynQuantMatMulDequant(x, B, bz, ws), plain)
    assert same_f32(rt.DynQuantMatMulDequant(x, B, bz, ws, bias), plain + bias)
    acts = [rt.DynQuantMatMulDequant(x, B, bz, ws, b, activation=a) for b in (None, bias) for a in (1, rt.ACTIVATION_GELU)]
    assert "split" in rt.last_gemm_kernel()
    monkeypatch.setenv("OM_MI355X_GEMM_TILE", "1")
    want = [rt.DynQuantMatMulDequant(x, B, bz, ws, b, activation=a) for b in (None, bias) for a in (1, rt.ACTIVATION_GELU)]
    assert "split" not in rt.last_gemm_kernel()
    monkeypatch.delenv("OM_MI355X_GEMM_TILE")
    assert all(same_f32(g, w) for g, w in zip(acts, want))
    # the result one element into a buffer, between guards
    whole, dA, dB = (rt.DeviceArray.from_numpy(v) for v in (np.full(1026 + M * N, 0x5A5A5A5A, np.int32), A, B))
    rt.MatMulInteger(dA, dB, None, None, out=rt.DeviceArray.view_of(whole, 513, (M, N)))
    assert "split" in rt.last_gemm_kernel()
    rt.synchronize()
    got = whole.numpy()
    assert np.array_equal(got[513:-513].reshape(M, N), mm(oracle, A, B, None, None))
    assert np.all(got[:513] == 0x5A5A5A5A) and np.all(got[-513:] == 0x5A5A5A5A)


@pytest.mark.parametrize("M,K,N,split", [(300, 1152, 260, False), (4096, 1280, 768, False), (300, 2048, 130, True)])
def test_whole_k_steps_take_the_form_without_a_tail(rt, oracle, M, K, N, split):
    """k_gemm_i8_dma: only a K that ends inside a step takes the form that looks
    for the end of the row in every step; both against the oracle, with row sums."""
    rng = np.random.default_rng(K)
    for k, ragged in ((K, False), (K + 16, True), (K + 48, True), (K + 64, False)):
        A, B = _rand_q(rng, np.uint8, (M, k)), _rand_q(rng, np.int8, (k, N))
        az, bz = _rand_q(rng, np.uint8, (1,)), _rand_q(rng, np.int8, (N,))
        assert np.array_equal(rt.MatMulInteger(A, B, az, bz), mm(oracle, A, B, az, bz))
        name = rt.last_gemm_kernel()
        assert "dma" in name and ("ragged" in name) == ragged and ("split" in name) == split, name


@pytest.mark.parametrize("M", [3, 9, 20, 40, 60])
def test_few_rows_row_sums_of_padded_steps(rt, oracle, M):
    """The weight-streaming kernel's row sums leave out the chunks it reads as
    zeros: steps that fill up a wave's last batch, and chunks past K.  Every K of
    whole chunks up to three steps a wave, and some beyond."""
    rng = np.random.default_rng(M)
    for K in list(range(16, 1600, 80)) + [1536, 2064, 2688, 5520]:
        A, B = rng.integers(0, 256, (M, K)).astype(np.uint8), rng.integers(0, 256, (K, 24)).astype(np.uint8)
        az, bz = np.uint8(121), rng.integers(0, 256, (24,)).astype(np.uint8)
        assert np.array_equal(rt.MatMulInteger(A, B, az, bz), oracle.matmul_integer(A, B, az, bz)), K


@pytest.mark.parametrize("M,K,N,layer,product", [
    (4, 2688, 5120, "quantized in the kernel, 2 x 16 columns", "(16 columns)"),
    (4, 8192, 4096, "quantized in the kernel, 16 columns", "directly"), (4, 8192, 4112, "quantized in the kernel, 16 columns", "(16 columns)"),
    (2, 2048, 4112, "quantized in the kernel, 2 x 16 columns", "directly"), (5, 4096, 5120, "quantized in the kernel, 2 x 16", "(16 columns)"),
    (4, 4096, 5120, "quantized in the kernel, 16 columns", "(16 columns)"), (8, 1536, 4608, "quantized in the kernel, 2 x 16", "(16 columns)"),
    (24, 256, 1024, "quantized in the kernel, 16 columns", "(16 columns)"), (24, 512, 5120, "quantized in the kernel, 2 x 16", "(32 columns)"),
    (24, 1536, 5120, "(32 columns)", "(32 columns)"), (24, 4096, 4112, "(16 columns)", "(16 columns)"), (24, 11008, 4096, "(16 columns)", "(16 columns)")])
def test_few_rows_tile_choice(rt, oracle, M, K, N, layer, product):
    """The weight-streaming kernel's tiles where each was measured to be the
    faster one (the choice had been carried over from one kind of operand to
    the others, up to a quarter slower); results against the oracle."""
    rng = np.random.default_rng(K + N)
    B, bz = rng.integers(-127, 128, (K, N)).astype(np.int8), rng.integers(-9, 9, (N,)).astype(np.int8)
    x, ws = rng.standard_normal((M, K), dtype=np.float32), rng.uniform(1e-3, 1e-2, N).astype(np.float32)
    q, s, z = oracle.dynamic_quantize_linear(x)
    want = oracle.matmul_integer(q, B, z, bz)
    got = rt.DynQuantMatMulDequant(x, B, bz, ws)
    assert layer in rt.last_gemm_kernel(), rt.last_gemm_kernel()
    assert same_f32(got, oracle.dequant_epilogue(want, s, ws))
    got = rt.MatMulInteger(q, B, z, bz)
    assert product in rt.last_gemm_kernel(), rt.last_gemm_kernel()
    assert np.array_equal(got, want)


@pytest.mark.parametrize("count,M,K,N,shared,one_launch", [
    (1, 1, 8192, 128, False, False), (1, 16, 4096, 1024, False, False), (1, 64, 2048, 128, False, False), (4, 1, 8192, 128, False, False),
    (2, 33, 8192, 100, True, False), (1, 130, 4096, 128, False, False), (3, 8, 4099, 130, False, True), (8, 1, 4096, 128, False, True),
    (1, 16, 128, 1024, False, True), (32, 33, 1024, 64, True, True), (3, 130, 512, 130, False, True)])
def test_batched_products_of_few_entries(rt, oracle, count, M, K, N, shared, one_launch):
    """A batched right-hand side with few entries and a long K goes to the kernels
    that split K over waves (one launch of few blocks took up to five times as
    long); either way the products are the oracle's, zero points per tensor and
    per matrix."""
    rng = np.random.default_rng(K + N + count)
    A, B = _rand_q(rng, np.uint8, (count, M, K)), _rand_q(rng, np.int8, (1 if shared else count, K, N))
    for az, bz in ((_rand_q(rng, np.uint8, ()), _rand_q(rng, np.int8, ())),
                   (_rand_q(rng, np.uint8, A.shape[:2] + (1,)), _rand_q(rng, np.int8, B.shape[:1] + (1, N)))):
        got = rt.MatMulInteger(A, B, az, bz)
        assert (rt.last_gemm_kernel() == "k_gemm_i8_batched") == one_launch, rt.last_gemm_kernel()
        for e in range(count):
            eb = 0 if shared else e
            za, zb = (az, bz) if az.ndim == 0 else (az[e].reshape(M), bz[eb].reshape(N))
            assert np.array_equal(got[e], mm(oracle, A[e], B[eb], np.atleast_1d(za), np.atleast_1d(zb))), e


def test_batched_products_matrix_by_matrix(rt):
    """More batch dimensions that alternate between the operands than one launch
    addresses: packed and multiplied matrix by matrix, the operands' matrices and
    zero points found through every dimension's stride."""
    rng = np.random.default_rng(5)
    M, K, N = 5, 48, 20
    A, B = _rand_q(rng, np.uint8, (2, 1, 2, 1, 3, M, K)), _rand_q(rng, np.int8, (1, 2, 1, 3, 1, K, N))
    az, bz = _rand_q(rng, np.uint8, A.shape[:-1] + (1,)), _rand_q(rng, np.int8, B.shape[:-2] + (1, N))
    for za, zb in ((None, None), (az, bz)):
        got = rt.MatMulInteger(A, B, za, zb)
        assert rt.last_gemm_kernel() != "k_gemm_i8_batched"
        a64, b64 = (v.astype(np.int64) - (0 if z is None else z.astype(np.int64)) for v, z in ((A, za), (B, zb)))
        assert np.array_equal(got, np.matmul(a64, b64))


def test_batched_products_in_two_launches(rt):
    """More blocks than one launch takes (2^20 entries of 5 tiles): the second
    launch's entries start where the first one's end."""
    rng = np.random.default_rng(6)
    E, M = 1 << 20, 257
    A, B = rng.integers(0, 256, (E, M, 1), np.uint8), rng.integers(-128, 128, (E, 1, 1), np.int8)
    got = rt.MatMulInteger(A, B, np.uint8(7), np.int8(-3))
    assert rt.last_gemm_kernel() == "k_gemm_i8_batched"
    for at in range(0, E, 1 << 17):
        part = slice(at, at + (1 << 17))
        assert np.array_equal(got[part], (A[part].astype(np.int32) - 7) * (B[part].astype(np.int32) + 3)), at


@pytest.mark.parametrize("front", ["one short of a trip", "a trip", "one more", "two trips and a part"])
def test_dynamic_quantize_with_a_front_that_is_reduced_first(rt, oracle, front):
    """Tensors whose front does not fit on chip: 56 float4 for each of 512 threads
    per CU are kept, what lies in front is reduced in trips of three float4 a
    thread and quantized by a second launch.  The extremes lie in turn at the last
    element of the front, at the first kept one and in the front's last trip."""
    threads = rt.device_info()["cus"] * 512
    trip = 3 * threads
    n_front = {"one short of a trip": trip - 1, "a trip": trip, "one more": trip + 1, "two trips and a part": 2 * trip + 777}[front]
    n = (56 * threads + n_front) * 4 + n_front % 4
    rng = np.random.default_rng(n_front)
    x = rng.standard_normal(n, dtype=np.float32)
    for at in (4 * n_front - 1, 4 * n_front, 4 * (n_front - n_front % trip) - 5 if n_front > 2 * trip else 4 * n_front - 9):
        x[at], x[at + 2] = 11.0 + at % 3, -9.0
        wy, ws, wz = oracle.dynamic_quantize_linear(x)
        dy, ds, dz = rt.DynamicQuantizeLinear(rt.DeviceArray.from_numpy(x))
        rt.synchronize()
        assert ds.numpy().view(np.uint32) == np.float32(ws).view(np.uint32) and int(dz.numpy()) == int(wz)
        assert np.array_equal(dy.numpy(), wy), at
        x[at] = x[at + 2] = 0.5


def test_layer_whose_rows_do_not_fit_on_chip(rt, oracle):
    """The fused layer's rows, stored minus 128, when their front is quantized by a
    launch of its own."""
    rng = np.random.default_rng(3)
    K, N = 1024, 24
    M = (rt.device_info()["cus"] * 512 * 4 * 56) // K + 1111
    x, B = rng.standard_normal((M, K), dtype=np.float32), _rand_q(rng, np.int8, (K, N))
    ws = rng.uniform(1e-3, 1e-2, N).astype(np.float32)
    q, s, z = oracle.dynamic_quantize_linear(x)
    assert same_f32(rt.DynQuantMatMulDequant(x, B, None, ws), oracle.dequant_epilogue(mm(oracle, q, B, z, None), s, ws))


@pytest.mark.parametrize("M,K,N", [(129, 4096, 258), (65, 1537, 66)])
def test_gelu_of_a_product_split_along_k(rt, oracle, M, K, N):
    """k_sum_parts applies onnx.Gelu itself: against the oracle's Gelu of the
    exact product.  Tolerance: 4 units in the last place of erf (2^-22) times
    |0.5 x|, plus one rounding of the result."""
    rng = np.random.default_rng(K)
    x, B = rng.normal(0, 1, (M, K)).astype(np.float32), _rand_q(rng, np.int8, (K, N))
    ws, bias = rng.uniform(1e-5, 1e-3, N).astype(np.float32), rng.normal(0, 1, N).astype(np.float32)
    q, s, z = oracle.dynamic_quantize_linear(x)
    plain = oracle.dequant_epilogue(mm(oracle, q, B, z, None), s, ws)
    for b, p in ((None, plain), (bias, plain + bias)):
        got = rt.DynQuantMatMulDequant(x, B, None, ws, b, activation=rt.ACTIVATION_GELU)
        assert "split" in rt.last_gemm_kernel(), rt.last_gemm_kernel()
        want = oracle.gelu(p).astype(np.float64)
        tol = np.abs(0.5 * p.astype(np.float64)) * 2.0 ** -22 + np.abs(want) * 2.0 ** -23 + 1e-45
        assert (np.abs(got - want) <= tol).all()
