"""MatMulInteger, its fused dequantising epilogue and QLinearMatMul on the GPU: integers exact,
floats bit for bit (the epilogue rounds twice, like the unfused Cast, Mul, Add)."""
import json
import os

import numpy as np
import pytest

import refcases as rc

pytestmark = pytest.mark.gpu


def test_reference_variants_cases(ctx, pkg, oracle):
    """crates/onnx-vulkan-core/tests/matmul_integer_variants.rs:113-137, 174-196, 255-282."""
    a = rc.pseudo_plus1(7 * 12, 11).reshape(7, 12)
    b = rc.pseudo_plus1(12 * 5, 29).reshape(12, 5)
    assert np.array_equal(pkg.ops.matmul_integer(ctx, a, b, 37, 211), rc.matmul_integer_bigint(a, b, 37, 211))
    for (m, k, n) in [(20, 64, 18), (150, 96, 90)]:
        a = rc.pseudo_plus1(m * k, 3).reshape(m, k)
        b = rc.pseudo_plus1(k * n, 41).reshape(k, n)
        assert np.array_equal(pkg.ops.matmul_integer(ctx, a, b, 37, 211), oracle.matmul_integer(a, b, 37, 211))
        bi = b.view(np.int8)
        assert np.array_equal(pkg.ops.matmul_integer(ctx, a, bi, 37, -73), oracle.matmul_integer(a, bi, 37, -73))


def test_as_a_node_with_leading_dimensions(ctx, pkg, oracle):
    a = rc.pseudo_plus1(2 * 50 * 64, 1).reshape(2, 50, 64)
    w = rc.pseudo_plus1(64 * 200, 2).view(np.int8).reshape(64, 200)
    node = pkg.graph.NodeIr("MatMulInteger", ["a", "w", "a_zp", "w_zp"], ["acc"])
    env = {"a": a, "w": w, "a_zp": np.array(131, np.uint8), "w_zp": np.array(-7, np.int8)}
    pkg.graph.execute(ctx, [node], env)
    assert env["acc"].shape == (2, 50, 200) and env["acc"].dtype == np.int32
    assert np.array_equal(env["acc"].reshape(100, 200), oracle.matmul_integer(a.reshape(100, 64), w, 131, -7))
    with pytest.raises(ValueError):
        pkg.graph.execute(ctx, [node], dict(env, w=w[:60]))


@pytest.mark.parametrize("a_dt,b_dt", [(np.uint8, np.int8), (np.uint8, np.uint8), (np.int8, np.int8), (np.int8, np.uint8)])
@pytest.mark.parametrize("shape", [(1, 4, 1), (3, 2, 5), (33, 49, 130), (130, 100, 257), (7, 1000, 3), (256, 128, 128)],
                         ids=lambda s: "M%d_K%d_N%d" % s)
def test_any_k_any_sign(ctx, pkg, oracle, shape, a_dt, b_dt):
    """K not a multiple of 4 or 16, tiles with ragged edges, all four sign combinations
    (tests/matmul_integer_any_k.rs:141-150)."""
    m, k, n = shape
    a = rc.pseudo_plus1(m * k, 5).view(a_dt).reshape(m, k)
    b = rc.pseudo_plus1(k * n, 6).view(b_dt).reshape(k, n)
    za = -9 if a_dt == np.int8 else 200
    zb = 17 if b_dt == np.int8 else 3
    want = oracle.matmul_integer(a, b, za, zb)
    assert np.array_equal(pkg.ops.matmul_integer(ctx, a, b, za, zb), want)
    assert np.array_equal(pkg.ops.matmul_integer(ctx, a, b, za, zb, raw=True), want)
    assert np.array_equal(pkg.ops.matmul_integer(ctx, a, b, None, None), oracle.matmul_integer(a, b, 0, 0))


@pytest.mark.parametrize("shape", [(1000, 1024, 4096), (1000, 4096, 1024)], ids=lambda s: "M%d_K%d_N%d" % s)
def test_ffn_pair_shapes(ctx, pkg, oracle, shape):
    """The dynamic int8 FFN pair: DynamicQuantizeLinear output times symmetric int8 weights."""
    m, k, n = shape
    x = pkg.synth.normal_f32(m * k, 21).reshape(m, k)
    a, a_scale, a_zp = pkg.ops.dynamic_quantize_linear(ctx, x)
    w = pkg.synth.int8_weight(k, n, 22)
    want = oracle.matmul_integer(a, w, a_zp, 0)
    weight = pkg.ops.Int8Weight(ctx, w)
    got = pkg.ops.matmul_integer(ctx, a, w, a_zp, 0, weight=weight)
    assert np.array_equal(got, want)
    # "then fp32 rescale": scale = a_scale * w_scale formed by the fused node, bias per column
    w_scale = np.float32(0.01)
    bias = pkg.synth.uniform_f32(n, 23, -0.5, 0.5)
    got = pkg.ops.matmul_integer_scale_bias(ctx, a, w, a_zp, 0, a_scale, bias, product=w_scale, weight=weight)
    ref = oracle.rescale(want, a_scale, bias, product=w_scale)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
    weight.destroy()


@pytest.mark.parametrize("a_dt,b_dt", [(np.uint8, np.int8), (np.int8, np.uint8)])
def test_large_products_take_the_256x256_tiles(ctx, pkg, oracle, a_dt, b_dt):
    """Enough 256x256 tiles to fill the chip switches to the large tile of the kernel that keeps B out of
    LDS: ragged edges in both directions, an odd number of k stages, both zero points non-zero, then the
    same product through the float epilogue."""
    m, k, n = 3601, 384, 3585
    a = rc.pseudo_plus1(m * k, 31).view(a_dt).reshape(m, k)
    b = rc.pseudo_plus1(k * n, 32).view(b_dt).reshape(k, n)
    za = -9 if a_dt == np.int8 else 200
    zb = 17 if b_dt == np.int8 else 3
    want = oracle.matmul_integer(a, b, za, zb)
    weight = pkg.ops.Int8Weight(ctx, b)
    assert np.array_equal(pkg.ops.matmul_integer(ctx, a, b, za, zb, weight=weight), want)
    scale = np.float32(0.003)
    bias = pkg.synth.uniform_f32(n, 33, -0.5, 0.5)
    got = pkg.ops.matmul_integer_scale_bias(ctx, a, b, za, zb, scale, bias, weight=weight)
    assert np.array_equal(got.view(np.uint32), oracle.rescale(want, scale, bias).view(np.uint32))
    weight.destroy()


@pytest.mark.parametrize("a_dt,b_dt", [(np.uint8, np.int8), (np.uint8, np.uint8), (np.int8, np.int8), (np.int8, np.uint8)])
@pytest.mark.parametrize("shape", [(130, 640, 257), (70, 1536, 64), (1, 512, 1), (333, 4096, 200)], ids=lambda s: "M%d_K%d_N%d" % s)
def test_few_tiles_and_long_k_take_the_k_split_kernel(ctx, pkg, oracle, shape, a_dt, b_dt):
    """Up to two 64x64 tiles per CU with k a multiple of 128 and at least 512: the workgroup's
    wavefronts split k, A alone passes through LDS, B comes fragment by fragment from the
    fragment-major prepacked weight. Stage counts that are not a multiple of the four in flight
    (5, 12, 4, 32), ragged edges, zero points on both sides or none, and the float epilogue."""
    m, k, n = shape
    a = rc.pseudo_plus1(m * k, 51).view(a_dt).reshape(m, k)
    b = rc.pseudo_plus1(k * n, 52).view(b_dt).reshape(k, n)
    za = -9 if a_dt == np.int8 else 200
    zb = 17 if b_dt == np.int8 else 3
    want = oracle.matmul_integer(a, b, za, zb)
    weight = pkg.ops.Int8Weight(ctx, b)
    assert np.array_equal(pkg.ops.matmul_integer(ctx, a, b, za, zb, weight=weight), want)
    assert np.array_equal(pkg.ops.matmul_integer(ctx, a, b, None, None, weight=weight), oracle.matmul_integer(a, b, 0, 0))
    scale = np.float32(0.002)
    bias = pkg.synth.uniform_f32(n, 53, -0.5, 0.5)
    got = pkg.ops.matmul_integer_scale_bias(ctx, a, b, za, zb, scale, bias, weight=weight)
    assert np.array_equal(got.view(np.uint32), oracle.rescale(want, scale, bias).view(np.uint32))
    weight.destroy()


LAYERS = [  # tests/matmul_integer_epilogue.rs:352-420: (a_shape, N, weight int8?, relu, per-column scale)
    ((2, 50, 64), 200, False, False, False), ((700, 96), 330, True, False, False),
    ((1100, 64), 1040, False, True, False), ((1, 128, 32), 48, True, False, True),
    ((5, 70), 9, True, True, True),      # K % 4 != 0, fewer than 16 rows and columns
]


@pytest.mark.parametrize("layer", LAYERS, ids=lambda l: "x".join(map(str, l[0])) + "_N%d" % l[1])
def test_fused_epilogue_equals_cast_mul_add_bit_for_bit(ctx, pkg, oracle, layer):
    a_shape, n, w_signed, relu, per_col = layer
    k = a_shape[-1]
    m = int(np.prod(a_shape[:-1]))
    a = rc.pseudo_plus1(m * k, 1).reshape(m, k)
    w = rc.pseudo_plus1(k * n, 2).view(np.int8 if w_signed else np.uint8).reshape(k, n)
    a_zp, w_zp = 131, (-7 if w_signed else 121)
    a_scale = np.float32(0.0123)
    w_scale = pkg.synth.uniform_f32(n, 4, 1e-3, 5e-3) if per_col else np.float32(3.1e-3)
    bias = pkg.synth.uniform_f32(n, 3, -0.5, 0.5)
    acc = oracle.matmul_integer(a, w, a_zp, w_zp)
    ref = oracle.rescale(acc, a_scale, bias, product=w_scale, relu=relu)
    got, folded = pkg.ops.matmul_integer_scale_bias(ctx, a, w, a_zp, w_zp, a_scale, bias, product=w_scale, relu=relu,
                                                    fold_range=True)
    differing = int(np.count_nonzero(got.view(np.uint32) != ref.view(np.uint32)))
    assert differing == 0, f"{differing} of {got.size} elements differ"
    if relu:
        assert np.count_nonzero(got == 0) > got.size // 8
    # the folded range is the one a min/max pass over the result finds
    assert folded[0] == np.float32(-min(ref.min(), 0)).view(np.uint32) & 0x7FFFFFFF
    assert folded[1] == np.float32(max(ref.max(), 0)).view(np.uint32)
    # without a bias and with a scalar scale only
    got = pkg.ops.matmul_integer_scale_bias(ctx, a, w, a_zp, w_zp, a_scale)
    assert np.array_equal(got.view(np.uint32), oracle.rescale(acc, a_scale).view(np.uint32))


def test_a_folded_range_feeds_the_next_quantisation(ctx, pkg, oracle):
    """MatMulIntegerScaleBias(range) -> DynamicQuantizeLinear(range_ready) must give the bytes,
    scale and zero point of a DynamicQuantizeLinear with its own pass (matmul_integer_epilogue.rs:1-12)."""
    m, k, n = 300, 128, 260
    a = rc.pseudo_plus1(m * k, 9).reshape(m, k)
    w = rc.pseudo_plus1(k * n, 10).view(np.int8).reshape(k, n)
    weight = pkg.ops.Int8Weight(ctx, w)
    dA, dza = ctx.upload(a), ctx.upload(np.array([128], np.uint8))
    dS = ctx.upload(np.array([0.004], np.float32))
    dY, dR, dQ, dP = ctx.alloc(m * n * 4), ctx.alloc(8), ctx.alloc(m * n), ctx.alloc(8)
    ctx.fill(dR, 0, 8, 0)
    pkg.ops.matmul_integer_scale_bias_device(ctx, dA, pkg.U8, weight, dza, None, dS, 0, None, 0, None, 0, False, dR, dY, m)
    pkg.ops.dynamic_quantize_linear_device(ctx, dY, m * n, dQ, dP, dP.at(4), range_slot=dR, range_ready=True)
    y = oracle.rescale(oracle.matmul_integer(a, w, 128, 0), np.float32(0.004))
    wq, ws, wz = oracle.dynamic_quantize_linear(y)
    assert np.array_equal(ctx.download(dQ, np.uint8, (m, n)), wq)
    assert ctx.download(dP, np.float32, (1,))[0].tobytes() == np.float32(ws).tobytes()
    assert ctx.download(dP, np.uint8, (1,), offset=4)[0] == wz
    weight.destroy()


def _golden():
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "qlinear_golden.json")
    with open(path) as f:
        return [c for c in json.load(f) if c["op"] == "QLinearMatMul"]


@pytest.mark.parametrize("case", _golden(), ids=lambda c: c["name"])
def test_qlinear_matmul_golden_literals(ctx, pkg, case):
    node = pkg.graph.NodeIr("QLinearMatMul", ["a", "a_scale", "a_zp", "b", "b_scale", "b_zp", "y_scale", "y_zp"], ["out"])
    env = {"a": np.array(case["a"], np.uint8).reshape(case["a_shape"]), "a_scale": np.float32(case["a_scale"]),
           "a_zp": np.array(case["a_zp"], np.uint8), "b": np.array(case["b"], np.int8).reshape(case["b_shape"]),
           "b_scale": np.array(case["b_scale"], np.float32), "b_zp": np.array(case["b_zp"], np.int8),
           "y_scale": np.float32(case["y_scale"]), "y_zp": np.array(case["y_zp"], np.uint8)}
    pkg.graph.execute(ctx, [node], env)
    assert env["out"].reshape(-1).tolist() == case["want"]


@pytest.mark.parametrize("per_col", [False, True])
@pytest.mark.parametrize("y_signed", [False, True])
def test_qlinear_matmul_seeded(ctx, pkg, oracle, per_col, y_signed):
    m, k, n = 77, 200, 150
    a = rc.pseudo_plus1(m * k, 12).reshape(m, k)
    b = rc.pseudo_plus1(k * n, 13).view(np.int8).reshape(k, n)
    b_scale = pkg.synth.uniform_f32(n, 14, 0.001, 0.02) if per_col else np.float32(0.01)
    b_zp = 0 if per_col else 5
    y_zp = -3 if y_signed else 120
    got = pkg.ops.qlinear_matmul(ctx, a, 0.02, 128, b, b_scale, b_zp, 0.9, y_zp, y_signed)
    want = oracle.qlinear_matmul(a, 0.02, 128, b, b_scale, b_zp, 0.9, y_zp, y_signed)
    assert np.max(np.abs(got.astype(int) - want.astype(int))) <= 1     # the stated +-1 LSB ...
    assert np.array_equal(got, want)                                   # ... and in fact identical
    assert 0.2 < np.mean((got != got.max()) & (got != got.min())), "the case must not saturate everywhere"


def test_qlinear_matmul_refuses_asymmetric_per_column_weights(ctx, pkg):
    a = np.zeros((4, 16), np.uint8)
    b = np.zeros((16, 8), np.int8)
    with pytest.raises(pkg.HipComputeError) as e:
        pkg.ops.qlinear_matmul(ctx, a, 0.02, 128, b, np.full(8, 0.01, np.float32), 3, 0.05, 10)
    assert e.value.code == 2 and "per-channel zero point" in e.value.message
    with pytest.raises(pkg.HipComputeError) as e:
        pkg.ops.qlinear_matmul(ctx, a, 0.02, 128, b, np.full(5, 0.01, np.float32), 0, 0.05, 10)
    assert e.value.code == 1


def test_requantize_alone(ctx, pkg, oracle):
    acc = pkg.synth.uniform_ints(3 * 7 * 11, 15, -90000, 90000).astype(np.int32).reshape(3, 7, 11)
    ratio = pkg.synth.uniform_f32(7, 16, 0.0005, 0.003)
    bias = pkg.synth.uniform_ints(7, 17, -5000, 5000).astype(np.int32)
    for signed, zp in [(False, 100), (True, -20)]:
        got = pkg.ops.requantize(ctx, acc, bias, ratio, 11, zp, signed)
        assert np.array_equal(got, oracle.requantize(acc, bias, ratio, 11, zp, signed))
    got = pkg.ops.requantize(ctx, acc.reshape(-1)[:229], None, ratio[:1], 1, 7, False)   # ragged tail, scalar ratio
    assert np.array_equal(got, oracle.requantize(acc.reshape(-1)[:229], None, ratio[:1], 1, 7, False))


SIGNS = [(np.uint8, np.int8), (np.uint8, np.uint8), (np.int8, np.int8), (np.int8, np.uint8)]


def _mm_three_epilogues(ctx, pkg, oracle, m, k, n, a_dt, b_dt, seed):
    """int32, rescaled float and requantised byte outputs of one product against the oracle."""
    a = rc.pseudo_plus1(m * k, seed).view(a_dt).reshape(m, k)
    b = rc.pseudo_plus1(k * n, seed + 1).view(b_dt).reshape(k, n)
    za = -9 if a_dt == np.int8 else 200
    zb = 17 if b_dt == np.int8 else 3
    want = oracle.matmul_integer(a, b, za, zb)
    weight = pkg.ops.Int8Weight(ctx, b)
    assert np.array_equal(pkg.ops.matmul_integer(ctx, a, b, za, zb, weight=weight), want)
    scale = np.float32(0.003)
    bias = pkg.synth.uniform_f32(n, seed + 2, -0.5, 0.5)
    got = pkg.ops.matmul_integer_scale_bias(ctx, a, b, za, zb, scale, bias, relu=True, weight=weight)
    assert np.array_equal(got.view(np.uint32), oracle.rescale(want, scale, bias, relu=True).view(np.uint32))
    ys = float(0.02 * 0.01 * 74 * 73 * np.sqrt(k) / 100.0)
    got = pkg.ops.qlinear_matmul(ctx, a, 0.02, za, b, np.float32(0.01), zb, ys, 7, True, weight=weight)
    assert np.array_equal(got, oracle.qlinear_matmul(a, 0.02, za, b, np.float32(0.01), zb, ys, 7, True))
    weight.destroy()


@pytest.mark.parametrize("a_dt,b_dt", SIGNS)
@pytest.mark.parametrize("shape", [(2048, 384, 4096), (2017, 200, 4001), (3000, 256, 3000)], ids=lambda s: "M%d_K%d_N%d" % s)
def test_many_tiles_take_the_128x128_kernel(ctx, pkg, oracle, shape, a_dt, b_dt):
    """192 or more 128x128 tiles but fewer than 192 of 256x256: with whole 128-byte k stages the 128x128
    tile of the kernel that keeps B out of LDS (three stages, then an even count), with k = 200 and
    ragged rows and columns the LDS-staged 128x128 kernel in its unaligned form; every sign
    combination, both zero points non-zero, all three epilogues."""
    m, k, n = shape
    _mm_three_epilogues(ctx, pkg, oracle, m, k, n, a_dt, b_dt, seed=61)


ROUTES = [  # (options, M, K, N): every alternative route of the integer product once, forced in process
    ({"HIPC_GEMM_TILE": 128, "HIPC_GEMM_BIG": 0, "HIPC_GEMM_SMALL": 0}, 300, 640, 260),
    ({"HIPC_GEMM_TILE": 64, "HIPC_GEMM_BIG": 0, "HIPC_GEMM_SMALL": 0}, 1000, 1024, 520),
    ({"HIPC_GEMM_BIG": 1}, 700, 384, 520),                  # B out of LDS, 256x256 tiles: ragged, three stages
    ({"HIPC_GEMM_BIG": 2}, 333, 128, 390),                  # ... 128x128 tiles: ragged, a single stage
    ({"HIPC_GEMM_BIG": 2}, 1000, 1024, 4096),               # ... the first product of the dynamic int8 FFN
    ({"HIPC_GEMM_SMALL": 1, "HIPC_GEMM_BIG": 0}, 2100, 256, 1030),
    ({"HIPC_GEMM_SMALL": 0, "HIPC_GEMM_BIG": 0}, 1000, 1024, 1024),
]


@pytest.mark.parametrize("options,m,k,n", ROUTES, ids=lambda v: str(v).replace(" ", "") if isinstance(v, dict) else str(v))
def test_every_route_of_the_integer_product_can_be_forced(ctx, pkg, oracle, options, m, k, n):
    with ctx.options(**options):
        _mm_three_epilogues(ctx, pkg, oracle, m, k, n, np.uint8, np.int8, seed=71)
        _mm_three_epilogues(ctx, pkg, oracle, m, k, n, np.int8, np.uint8, seed=73)


@pytest.mark.parametrize("route", [dict(HIPC_GEMM_BIG=1), dict(HIPC_GEMM_BIG=2), dict(HIPC_GEMM_BIG=0, HIPC_GEMM_SMALL=1),
                                   dict(HIPC_GEMM_BIG=0, HIPC_GEMM_SMALL=0, HIPC_GEMM_TILE=64),
                                   dict(HIPC_GEMM_BIG=0, HIPC_GEMM_SMALL=0, HIPC_GEMM_TILE=128)],
                         ids=["tile256", "tile128", "k_split", "staged64", "staged128"])
@pytest.mark.parametrize("shape", [(133, 16, 70), (70, 112, 140), (257, 400, 131), (129, 1424, 260), (66, 1001, 130), (131, 127, 64)],
                         ids=lambda s: "M%d_K%d_N%d" % s)
def test_rows_that_are_not_whole_stages(ctx, pkg, oracle, shape, route):
    """K a multiple of 16 but not of a stage's 128 (the last stage reads the row's end), and K that is not (the rows are
    copied to a pitch that is); zero points on both sides, so that the sums over A's rows count, and none."""
    m, k, n = shape
    a = rc.pseudo_plus1(m * k, 61).reshape(m, k)
    for b, za, zb in ((rc.pseudo_plus1(k * n, 62).reshape(k, n), 200, 3), (rc.pseudo_plus1(k * n, 63).view(np.int8).reshape(k, n), 131, None)):
        want = oracle.matmul_integer(a, b, za, zb or 0)
        with ctx.options(**route):
            assert np.array_equal(pkg.ops.matmul_integer(ctx, a, b, za, zb), want)


@pytest.mark.parametrize("shape", [(70, 16, 7), (65, 128, 64), (64, 144, 130), (129, 256, 131), (257, 1040, 65), (70, 1136, 190), (133, 1280, 260)],
                         ids=lambda s: "M%d_K%d_N%d" % s)
def test_two_groups_share_the_stages(ctx, pkg, oracle, shape):
    """64x64 tiles whose stages two groups of wavefronts take in turn: fewer stages than groups, an odd count (one group's last is
    past the end), one more than a group has in flight; ragged tiles; sums over A's rows; every epilogue."""
    m, k, n = shape
    with ctx.options(HIPC_GEMM_BIG=0, HIPC_GEMM_SMALL=2):
        _mm_three_epilogues(ctx, pkg, oracle, m, k, n, np.uint8, np.int8, seed=75)
        _mm_three_epilogues(ctx, pkg, oracle, m, k, n, np.int8, np.uint8, seed=77)
        a, b = rc.pseudo_plus1(m * k, 78).reshape(m, k), rc.pseudo_plus1(k * n, 79).view(np.int8).reshape(k, n)
        assert np.array_equal(pkg.ops.matmul_integer(ctx, a, b, 131, None), oracle.matmul_integer(a, b, 131, 0))


@pytest.mark.parametrize("offset,k", [(4, 256), (3, 128), (1, 45), (2, 16)])
def test_rows_at_any_address(ctx, pkg, oracle, offset, k):
    """A inside a larger buffer, at an address that is not a multiple of 16 (or of 4)."""
    m, n = 37, 75
    a = rc.pseudo_plus1(m * k, 64).reshape(m, k)
    b = rc.pseudo_plus1(k * n, 65).view(np.int8).reshape(k, n)
    weight = pkg.ops.Int8Weight(ctx, b)
    buf, y, z = ctx.alloc(m * k + offset), ctx.alloc(m * n * 4), ctx.upload(np.array([9, 5], np.uint8))
    ctx.upload(a, buf, offset)
    pkg.ops.matmul_integer_device(ctx, buf.at(offset), pkg.U8, weight, z.ptr, z.at(1), y, m)
    assert np.array_equal(ctx.download(y, np.int32, (m, n)), oracle.matmul_integer(a, b, 9, 5))
    weight.destroy()
    for x in (buf, y, z):
        x.free()


@pytest.mark.parametrize("route", [dict(HIPC_GEMM_BIG=1), dict(HIPC_GEMM_BIG=2), dict(HIPC_GEMM_BIG=0, HIPC_GEMM_SMALL=1), {}],
                         ids=["tile256", "tile128", "k_split", "chosen"])
@pytest.mark.parametrize("n", [272, 260, 131, 7])
@pytest.mark.parametrize("signed", [False, True])
def test_requantized_bytes_leave_as_rows(ctx, pkg, oracle, n, signed, route):
    """Output rows that are whole 16-byte pieces, whole words, neither; both output types; ratios that saturate."""
    m, k = 145, 144
    a = rc.pseudo_plus1(m * k, 71).reshape(m, k)
    b = rc.pseudo_plus1(k * n, 72).view(np.int8).reshape(k, n)
    b_scale = pkg.synth.uniform_f32(n, 73, 1e-4, 2e-2)
    zp = -5 if signed else 130
    want = oracle.qlinear_matmul(a, 0.02, 128, b, b_scale, 0, 0.05, zp, y_signed=signed)
    with ctx.options(**route):
        assert np.array_equal(pkg.ops.qlinear_matmul(ctx, a, 0.02, 128, b, b_scale, 0, 0.05, zp, y_signed=signed), want)


@pytest.mark.parametrize("b_dt", [np.int8, np.uint8])
@pytest.mark.parametrize("shape", [(1, 16, 1), (16, 128, 16), (17, 1008, 100), (32, 2064, 33), (33, 320, 8200), (64, 4096, 132), (5, 8208, 48)],
                         ids=lambda s: "M%d_K%d_N%d" % s)
def test_few_rows(ctx, pkg, oracle, shape, b_dt):
    """Up to 64 rows: 1, 2 and 4 blocks of 16 rows, one and two blocks of columns, 4 to 16 wavefronts along k with fewer
    steps than they have in flight and more than one round of them; int32, the folded range, bytes."""
    m, k, n = shape
    a = rc.pseudo_plus1(m * k, 81).reshape(m, k)
    b = rc.pseudo_plus1(k * n, 82).view(b_dt).reshape(k, n)
    want = oracle.matmul_integer(a, b, 131, 17)
    with ctx.options(HIPC_GEMM_SKINNY=1):
        weight = pkg.ops.Int8Weight(ctx, b)
        assert np.array_equal(pkg.ops.matmul_integer(ctx, a, b, 131, 17, weight=weight), want)
        bias = pkg.synth.uniform_f32(n, 83, -0.5, 0.5)
        got, folded = pkg.ops.matmul_integer_scale_bias(ctx, a, b, 131, 17, np.float32(0.002), bias, fold_range=True, weight=weight)
        ref = oracle.rescale(want, np.float32(0.002), bias)
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
        assert folded[0] == np.float32(-min(ref.min(), 0)).view(np.uint32) & 0x7FFFFFFF and folded[1] == np.float32(max(ref.max(), 0)).view(np.uint32)
        for signed in (False, True):
            assert np.array_equal(pkg.ops.qlinear_matmul(ctx, a, 0.02, 131, b, 0.01, 17, 0.5, 3, y_signed=signed, weight=weight),
                                  oracle.qlinear_matmul(a, 0.02, 131, b, 0.01, 17, 0.5, 3, y_signed=signed))
        weight.destroy()


@pytest.mark.parametrize("shape", [(17, 512, 1024), (33, 1100, 2048), (48, 64, 1366), (49, 4160, 500), (64, 1024, 2050), (64, 128, 4100)], ids=lambda s: "M%d_K%d_N%d" % s)
def test_few_rows_over_several_workgroups(ctx, pkg, oracle, shape):
    """One, two and all blocks of 16 rows to a workgroup, the last block of one row or of all, columns one past a block: int32
    and the folded range."""
    m, k, n = shape
    a = rc.pseudo_plus1(m * k, 84).reshape(m, k)
    b = rc.pseudo_plus1(k * n, 85).view(np.int8).reshape(k, n)
    want = oracle.matmul_integer(a, b, 131, 0)
    weight = pkg.ops.Int8Weight(ctx, b)
    with ctx.options(HIPC_GEMM_SKINNY=1):
        assert np.array_equal(pkg.ops.matmul_integer(ctx, a, b, 131, 0, weight=weight), want)
        bias = pkg.synth.uniform_f32(n, 86, -0.5, 0.5)
        got, folded = pkg.ops.matmul_integer_scale_bias(ctx, a, b, 131, 0, np.float32(0.002), bias, fold_range=True, weight=weight)
    weight.destroy()
    ref = oracle.rescale(want, np.float32(0.002), bias)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
    assert folded[0] == np.float32(-min(ref.min(), 0)).view(np.uint32) & 0x7FFFFFFF and folded[1] == np.float32(max(ref.max(), 0)).view(np.uint32)


@pytest.mark.parametrize("m,k,n", [(5, 256, 96), (40, 250, 200), (64, 128, 4096), (70, 249, 96), (300, 1000, 130), (600, 1001, 900), (2500, 250, 2600), (70, 4112, 130), (130, 4113, 260)])
def test_a_recorded_weight_zero_point_of_zero_can_be_patched(ctx, pkg, oracle, m, k, n):
    """A QLinearMatMul recorded with an int8 weight and zero point 0 -- few rows, rows that are no whole 16 bytes -- and
    replayed with others."""
    a = pkg.synth.uniform_ints(m * k, 801, 0, 255).astype(np.uint8).reshape(m, k)
    b = pkg.synth.int8_weight(k, n, 802)
    w = pkg.ops.Int8Weight(ctx, b)
    dA, dY = ctx.upload(a), ctx.alloc(m * n)
    ys = 0.02 * 0.01 * 74 * 73 * np.sqrt(k) / 40
    call = lambda: pkg.ops.qlinear_matmul_device(ctx, dA, pkg.U8, 0.02, 128, w, np.float32(0.01), 0, ys, 120, pkg.U8, dY, m)  # noqa: E731
    call()
    ctx.flush()
    ctx.capture_begin()
    call()
    graph = ctx.capture_end()
    rt = pkg.runtime
    now = {rt.SCALAR_A_ZERO_POINT: 128, rt.SCALAR_B_ZERO_POINT: 0, rt.SCALAR_Y_ZERO_POINT: 120}
    for which, value in ((None, 0), (rt.SCALAR_A_ZERO_POINT, 90), (rt.SCALAR_B_ZERO_POINT, 3), (rt.SCALAR_Y_ZERO_POINT, 90), (rt.SCALAR_A_ZERO_POINT, 128), (rt.SCALAR_B_ZERO_POINT, 0)):
        if which:
            ctx.graph_set_scalar(graph, 0, which, value)
            now[which] = value
        ctx.fill(dY, 0, m * n // 4 * 4, 0)
        ctx.graph_launch(graph)
        want = oracle.qlinear_matmul(a, 0.02, now[rt.SCALAR_A_ZERO_POINT], b, np.float32(0.01), now[rt.SCALAR_B_ZERO_POINT], ys, now[rt.SCALAR_Y_ZERO_POINT], False)
        assert np.array_equal(ctx.download(dY, np.uint8, (m, n)), want), (which, value)
    ctx.graph_destroy(graph)
    w.destroy()
    dA.free(), dY.free()
