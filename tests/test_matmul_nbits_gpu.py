"""MatMulNBits on the GPU against the oracle, through the C ABI.

Tolerance (the one the task states for this operator): |got - ref| <= atol + rtol * |ref| with
atol = 1e-3 and rtol = 1e-4 for f32 tensors, rtol = 1e-3 for f16 tensors.
"""
import numpy as np
import pytest

import refcases as rc

pytestmark = pytest.mark.gpu

ATOL, RTOL32, RTOL16 = 1e-3, 1e-4, 1e-3


def close(got, ref, rtol):
    got, ref = got.astype(np.float64), ref.astype(np.float64)
    return np.all(np.abs(got - ref) <= ATOL + rtol * np.abs(ref))


def worst(got, ref):
    return float(np.max(np.abs(got.astype(np.float64) - ref.astype(np.float64))))


@pytest.mark.parametrize("case", rc.MATMUL_NBITS_CASES, ids=lambda c: "M%d_K%d_N%d_bs%d" % c)
def test_reference_cases_as_nodes(ctx, pkg, oracle, case):
    """The seven cases of crates/onnx-vulkan-core/tests/matmul_nbits.rs, built as the reference
    builds them: one com.microsoft::MatMulNBits node, tensors by name."""
    m, k, n, bs = case
    a, nib, zp, scale = rc.matmul_nbits_case(m, k, n, bs)
    B, Z = pkg.synth.pack_nibbles(nib, bs), pkg.synth.pack_zero_points(zp)
    node = pkg.graph.NodeIr("MatMulNBits", ["a", "quant", "scales", "zp"], ["out"],
                            {"K": k, "N": n, "bits": 4, "block_size": bs}, domain="com.microsoft", name="mmnb")
    assert pkg.graph.is_implemented_node(node)
    env = {"a": a, "quant": B, "scales": scale.reshape(-1), "zp": Z}
    pkg.graph.execute(ctx, [node], env)
    want = oracle.matmul_nbits(a, B, scale.reshape(-1), Z, k, n, bs)
    got = env["out"]
    assert got.shape == (m, n) and got.dtype == np.float32
    assert close(got, want, RTOL32), worst(got, want)
    # and the reference's own bound against the mathematics
    f64 = rc.matmul_nbits_f64(a, nib, zp, scale, bs)
    assert np.all(np.abs(got - f64) <= 1e-4 * np.maximum(np.abs(f64), 1.0))


@pytest.mark.parametrize("case", [c for c in rc.MATMUL_NBITS_CASES if c[3] >= 32], ids=lambda c: "M%d_K%d_N%d_bs%d" % c)
def test_reference_cases_on_the_prepacked_path(ctx, pkg, oracle, case):
    m, k, n, bs = case
    a, nib, zp, scale = rc.matmul_nbits_case(m, k, n, bs)
    B, Z = pkg.synth.pack_nibbles(nib, bs), pkg.synth.pack_zero_points(zp)
    w = pkg.ops.NBitsWeight(ctx, B, scale.reshape(-1), Z, k, n, bs)
    got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, weight=w)
    w.destroy()
    want = oracle.matmul_nbits(a, B, scale.reshape(-1), Z, k, n, bs)
    assert close(got, want, RTOL32), worst(got, want)


SHAPES = [  # (M, K, N, block_size, with_zp)
    (1, 1152, 6912, 32, True),    # gemma3 up / gate projection
    (1, 6912, 1152, 32, True),    # down projection
    (1, 1152, 1024, 32, True), (1, 1024, 1152, 32, True), (1, 1152, 256, 32, True),
    (2, 2048, 2560, 128, False),  # qwen-style block 128 without zero points
    (4, 300, 100, 64, True),      # partial last block, N not a multiple of 16
    (5, 4096, 48, 256, True),
    (8, 1152, 512, 32, True), (9, 512, 80, 32, False), (16, 640, 96, 32, True),
    (17, 256, 64, 32, True),      # more than one group of 16 rows
    (3, 7000, 40, 32, True),      # K large enough to split across workgroups
    (8, 6912, 1152, 32, True),
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "M%d_K%d_N%d_bs%d_zp%d" % s)
def test_seeded_shapes_both_paths(ctx, pkg, oracle, shape):
    m, k, n, bs, with_zp = shape
    B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=100 + n, with_zp=with_zp)
    a = pkg.synth.normal_f32(m * k, 7).reshape(m, k)
    want = oracle.matmul_nbits(a, B, scales, zp, k, n, bs)
    got = pkg.ops.matmul_nbits(ctx, a, B, scales, zp, k, n, bs)
    assert close(got, want, RTOL32), ("direct", worst(got, want))
    w = pkg.ops.NBitsWeight(ctx, B, scales, zp, k, n, bs)
    got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, weight=w)
    w.destroy()
    assert close(got, want, RTOL32), ("gemv", worst(got, want))


@pytest.mark.parametrize("k,n,bs", [(208, 50, 16), (200, 33, 8), (240, 50, 24), (1000, 64, 40), (330, 17, 48)],
                         ids=lambda v: str(v))
def test_small_and_odd_block_sizes(ctx, pkg, oracle, k, n, bs):
    """The reference accepts every block_size that is a positive multiple of 8 (interp.rs:447-464); those
    below 32 or not a power of two run on the kernel that reads the ONNX layout. 13 blocks of 16: odd,
    zero-point rows off word boundaries; 8, 24, 40, 48: blocks that are no power of two, partial last block.
    A handle for such a weight keeps the tensors as they are (the caller's copies may go) and gives the
    same bits; one row, a few and more than 32 (no tiled kernel for them)."""
    B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=3)
    w = pkg.ops.NBitsWeight(ctx, B, scales, zp, k, n, bs)
    for m in (1, 3, 40):
        a = pkg.synth.normal_f32(m * k, 8 + m).reshape(m, k)
        got = pkg.ops.matmul_nbits(ctx, a, B, scales, zp, k, n, bs)
        assert close(got, oracle.matmul_nbits(a, B, scales, zp, k, n, bs), RTOL32)
        by_handle = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, weight=w)
        assert np.array_equal(by_handle, got)
    a16 = pkg.synth.normal_f32(5 * k, 9).reshape(5, k).astype(np.float16)
    B16, s16, _ = pkg.synth.nbits_weight(n, k, bs, seed=4, with_zp=False, scale_dtype=np.float16)
    w16 = pkg.ops.NBitsWeight(ctx, B16, s16, None, k, n, bs)
    got = pkg.ops.matmul_nbits(ctx, a16, None, None, None, k, n, bs, weight=w16)
    assert got.dtype == np.float16 and close(got, oracle.matmul_nbits(a16, B16, s16, None, k, n, bs), RTOL16)
    assert w.nbytes == B.size + 4 * scales.size + zp.size
    w.destroy(), w16.destroy()


@pytest.mark.parametrize("shape", [(1, 2048, 2560, 128), (6, 1024, 300, 32), (40, 512, 128, 128)],
                         ids=lambda s: "M%d_K%d_N%d_bs%d" % s)
def test_f16_tensors(ctx, pkg, oracle, shape):
    m, k, n, bs = shape
    B, scales, _ = pkg.synth.nbits_weight(n, k, bs, seed=5, with_zp=False, scale_dtype=np.float16)
    a = pkg.synth.normal_f32(m * k, 9).reshape(m, k).astype(np.float16)
    want = oracle.matmul_nbits(a, B, scales, None, k, n, bs)
    got = pkg.ops.matmul_nbits(ctx, a, B, scales, None, k, n, bs)
    assert got.dtype == np.float16 and close(got, want, RTOL16), ("direct", worst(got, want))
    w = pkg.ops.NBitsWeight(ctx, B, scales, None, k, n, bs)
    got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, weight=w)
    w.destroy()
    assert got.dtype == np.float16 and close(got, want, RTOL16), ("gemv", worst(got, want))


PREFILL = [  # (M, K, N, block_size, zero points): ragged tiles, partial last stage, every scale grouping
    (100, 1000, 200, 32, True), (130, 384, 131, 64, True), (257, 640, 96, 128, True), (64, 256, 1024, 256, False),
    (17, 72, 16, 32, True),
]


@pytest.mark.parametrize("shape", PREFILL, ids=lambda s: "M%d_K%d_N%d_bs%d_zp%d" % s)
def test_f16_rows_beyond_sixteen_run_the_tiled_kernel(ctx, pkg, oracle, shape):
    """A and the scales share one element type in MatMulNBits, so the scales are f16 here too."""
    m, k, n, bs, with_zp = shape
    B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=41, with_zp=with_zp, scale_dtype=np.float16)
    a = pkg.synth.normal_f32(m * k, 42).reshape(m, k).astype(np.float16)
    want = oracle.matmul_nbits(a, B, scales, zp, k, n, bs)
    w = pkg.ops.NBitsWeight(ctx, B, scales, zp, k, n, bs)
    got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, weight=w)
    w.destroy()
    assert got.dtype == np.float16 and close(got, want, RTOL16), worst(got, want)


WIDE_ROUTES = [  # the 128-row tiles, forced on shapes that would take 64x64: each kernel, alone and with k split over workgroups
    {"HIPC_PREFILL_TILE": 192}, {"HIPC_PREFILL_TILE": 192, "HIPC_PREFILL_SPLIT": 2}, {"HIPC_PREFILL_TILE": 128},
    {"HIPC_PREFILL_TILE": 128, "HIPC_PREFILL_SPLIT": 2},
    {"HIPC_PREFILL_TILE": 128, "HIPC_PREFILL_DIRECT": 0}, {"HIPC_PREFILL_TILE": 128, "HIPC_PREFILL_DIRECT": 0, "HIPC_PREFILL_SPLIT": 3},
    {"HIPC_PREFILL_TILE": 64}, {"HIPC_PREFILL_TILE": 64, "HIPC_PREFILL_DIRECT": 0},
    # two groups of four wavefronts per workgroup, each with half of k (a group without a trip of its own among them)
    {"HIPC_PREFILL_TILE": 192, "HIPC_PREFILL_GROUPS": 2}, {"HIPC_PREFILL_TILE": 128, "HIPC_PREFILL_GROUPS": 2},
    {"HIPC_PREFILL_TILE": 128, "HIPC_PREFILL_GROUPS": 2, "HIPC_PREFILL_SPLIT": 2}, {"HIPC_PREFILL_TILE": 128, "HIPC_PREFILL_GROUPS": 1},
    {"HIPC_PREFILL_TILE": 64, "HIPC_PREFILL_GROUPS": 2}, {"HIPC_PREFILL_TILE": 64, "HIPC_PREFILL_GROUPS": 1},
]


@pytest.mark.parametrize("options", WIDE_ROUTES, ids=lambda v: str(v).replace(" ", ""))
@pytest.mark.parametrize("shape", PREFILL + [(300, 1152, 392, 32, True), (129, 512, 260, 64, False)], ids=lambda s: "M%d_K%d_N%d_bs%d_zp%d" % s)
def test_both_wide_tile_kernels_on_ragged_shapes(ctx, pkg, oracle, shape, options):
    """The kernel that dequantises the weight in the registers of the wavefront that multiplies it (its k order
    inside a stage differs from memory order, for both operands alike) and the one that passes it through LDS:
    ragged rows and columns, a partial last stage, an odd stage count, every scale grouping, zero points."""
    m, k, n, bs, with_zp = shape
    B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=47, with_zp=with_zp, scale_dtype=np.float16)
    a = pkg.synth.normal_f32(m * k, 48).reshape(m, k).astype(np.float16)
    want = oracle.matmul_nbits(a, B, scales, zp, k, n, bs)
    w = pkg.ops.NBitsWeight(ctx, B, scales, zp, k, n, bs)
    with ctx.options(**options):
        got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, weight=w)
    w.destroy()
    assert got.dtype == np.float16 and close(got, want, RTOL16), worst(got, want)


@pytest.mark.parametrize("options", [{"HIPC_PREFILL_TILE": 192}, {"HIPC_PREFILL_TILE": 128}, {"HIPC_PREFILL_TILE": 128, "HIPC_PREFILL_GROUPS": 2}, {"HIPC_PREFILL_TILE": 64},
                                     {"HIPC_PREFILL_TILE": 64, "HIPC_PREFILL_DIRECT": 0}], ids=lambda v: str(v).replace(" ", ""))
@pytest.mark.parametrize("bs,dtype", [(32, np.float16), (128, np.float16), (64, np.float32)], ids=lambda v: str(getattr(v, "__name__", v)))
def test_block_scales_of_zero_and_of_very_different_size(ctx, pkg, oracle, bs, dtype, options):
    """The kernels that keep the weight out of LDS hold their accumulators in units of the open block's scale and
    rescale them when the next block opens: blocks whose scale is 0 (a block of zeros), 1000 times larger or 10000
    times smaller than their neighbours must come out as from the running total the other kernels keep (the
    64x64 tiles are in the list as that control), first block and last block included."""
    m, k, n = 96, 1024, 200
    B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=49, with_zp=True, scale_dtype=dtype)
    sc = scales.reshape(n, -1).copy()
    sc[:, ::3] = 0
    sc[:, 1::7] *= dtype(1000)
    sc[:, 2::5] *= dtype(1e-4)
    sc[5] = 0                      # a column of zeros
    sc[6, :-1] = 0                 # only the last block counts
    sc[7, 1:] = 0                  # only the first
    scales = sc.reshape(scales.shape)
    a = pkg.synth.normal_f32(m * k, 50).reshape(m, k).astype(dtype)
    w = pkg.ops.NBitsWeight(ctx, B, scales, zp, k, n, bs)
    with ctx.options(**options):
        got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, weight=w)
    w.destroy()
    assert np.all(got[:, 5] == 0)
    # Scales seven orders of magnitude apart make sums that cancel: against the float64 product, with the f32
    # accumulation's share stated in units of the row's largest result (the oracle itself is 4e-4 of it away; a
    # rescaled accumulator rounds once more per block than a running total does)
    nib, z = _unpack(B, zp, k, n, bs)
    f64 = rc.matmul_nbits_f64(a, nib, z, scales.reshape(n, -1), bs)
    big = np.abs(f64).max(axis=1, keepdims=True)
    err = np.abs(got.astype(np.float64) - f64)
    if dtype is np.float16:
        assert np.all(err <= 1e-3 + 1e-3 * np.abs(f64) + 1e-6 * big), float((err - 1e-3 * np.abs(f64)).max())
    else:   # f32 rows travel as two f16 rows (22 bits): as in the test of that route
        assert np.all(err <= 2e-5 * big + 1e-3), float((err / big).max())


@pytest.mark.parametrize("shape", [(100, 1000, 200, 32, True), (257, 640, 96, 128, False)], ids=lambda s: "M%d_K%d_N%d_bs%d_zp%d" % s)
def test_many_rows_on_the_onnx_layout_take_the_tiled_kernels(ctx, pkg, oracle, shape):
    """hipc_matmul_nbits (the reference's own calling convention: the ONNX tensors on every call) with more rows
    than the decode kernels take writes the tiled form into scratch memory and runs the kernels of the prepacked
    path: the same bits as a handle gives, f16 and f32 rows, twice in a row with different weights (the scratch
    block is reused)."""
    m, k, n, bs, with_zp = shape
    for seed, dtype in ((61, np.float32), (62, np.float16), (63, np.float32)):   # (scales in the activations' type, as the operator has them)
        B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=seed, with_zp=with_zp, scale_dtype=dtype)
        rows = pkg.synth.normal_f32(m * k, seed + 10).reshape(m, k).astype(dtype)
        w = pkg.ops.NBitsWeight(ctx, B, scales, zp, k, n, bs)
        got = pkg.ops.matmul_nbits(ctx, rows, B, scales, zp, k, n, bs)
        by_handle = pkg.ops.matmul_nbits(ctx, rows, None, None, None, k, n, bs, weight=w)
        w.destroy()
        assert got.dtype == dtype and np.array_equal(got, by_handle)
        want = oracle.matmul_nbits(rows, B, scales, zp, k, n, bs)
        assert close(got, want, RTOL32 if dtype == np.float32 else RTOL16), worst(got, want)


F32_PREFILL = [  # (M, K, N, block_size, zero points)
    (100, 1000, 200, 32, True), (130, 384, 131, 64, True), (257, 640, 96, 128, False), (33, 72, 16, 32, True),
    (512, 2048, 2560, 128, False),
]


F32_ROUTES = [  # the default; the two terms of a row in one accumulator (64 x 128 tiles and the larger ones, two k
    # groups per workgroup, k split over workgroups, 64 x 64 tiles); the kernel
    # with both operands in LDS, whose 2 M result rows a last launch adds up
    {}, {"HIPC_PREFILL_TILE": 128}, {"HIPC_PREFILL_TILE": 192}, {"HIPC_PREFILL_TILE": 128, "HIPC_PREFILL_GROUPS": 2},
    {"HIPC_PREFILL_TILE": 128, "HIPC_PREFILL_SPLIT": 2}, {"HIPC_PREFILL_TILE": 192, "HIPC_PREFILL_GROUPS": 2, "HIPC_PREFILL_SPLIT": 2},
    {"HIPC_PREFILL_TILE": 64}, {"HIPC_PREFILL_DIRECT": 0}, {"HIPC_PREFILL_DIRECT": 0, "HIPC_PREFILL_TILE": 128, "HIPC_PREFILL_SPLIT": 2},
]


@pytest.mark.parametrize("options", F32_ROUTES, ids=lambda v: str(v).replace(" ", ""))
@pytest.mark.parametrize("shape", F32_PREFILL, ids=lambda s: "M%d_K%d_N%d_bs%d_zp%d" % s)
def test_f32_rows_beyond_thirty_two_run_the_tiled_kernel(ctx, pkg, oracle, shape, options):
    """More than 32 rows of f32 activations (the reference's own element type, interp.rs:6455-6472) go through
    the tiled matrix-core kernel as two f16 rows each, scaled per row by a power of two: against the oracle at
    the operator's f32 tolerance, against the float64 product at 2e-5 of the row's largest output, and equal
    in quality to the decode kernel's route (the same rows, 16 at a time)."""
    m, k, n, bs, with_zp = shape
    B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=45, with_zp=with_zp)
    a = pkg.synth.normal_f32(m * k, 46).reshape(m, k)
    a[0] *= np.float32(3.0e7)      # a row far beyond the f16 range, one far below it, one of zeros
    a[1] *= np.float32(1.0e-9)
    a[2] = 0
    want = oracle.matmul_nbits(a, B, scales, zp, k, n, bs)
    w = pkg.ops.NBitsWeight(ctx, B, scales, zp, k, n, bs)
    with ctx.options(**options):
        got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, weight=w)
    by_rows = np.concatenate([pkg.ops.matmul_nbits(ctx, a[i:i + 16], None, None, None, k, n, bs, weight=w) for i in range(0, m, 16)])
    w.destroy()
    assert got.dtype == np.float32 and got.shape == (m, n)
    # rows 0 and 1 are out of the absolute tolerance's scale: compare them relative to their own size
    scale = np.maximum(np.abs(want).max(axis=1, keepdims=True), 1e-30)
    assert np.all(np.abs(got - want) <= (1e-3 + 1e-4 * np.abs(want)) * np.maximum(scale / np.abs(want[3:]).max(), 1e-30) + 1e-4 * scale), worst(got, want)
    nib, z = _unpack(B, zp if zp is not None else np.full((n, (-(-k // bs) + 1) // 2), 0x88, np.uint8), k, n, bs)
    f64 = rc.matmul_nbits_f64(a, nib, z, scales.reshape(n, -1), bs)
    big = np.abs(f64).max(axis=1, keepdims=True)
    assert np.all(np.abs(got - f64) <= 2e-5 * np.maximum(big, 1e-300)), float(np.max(np.abs(got - f64) / np.maximum(big, 1e-300)))
    assert np.all(np.abs(got - f64) <= np.abs(by_rows - f64).max(axis=1, keepdims=True) * 1.5 + 2e-6 * big)
    assert np.all(got[2] == 0)


@pytest.mark.parametrize("options", [{}, {"HIPC_PREFILL_TILE": 64}, {"HIPC_PREFILL_TILE": 128, "HIPC_PREFILL_GROUPS": 2}, {"HIPC_PREFILL_TILE": 192},
                                     {"HIPC_PREFILL_TILE": 128, "HIPC_PREFILL_SPLIT": 2}, {"HIPC_PREFILL_DIRECT": 0}], ids=lambda v: str(v).replace(" ", ""))
@pytest.mark.parametrize("level", [2, 3, 4])
@pytest.mark.parametrize("shape", F32_PREFILL, ids=lambda s: "M%d_K%d_N%d_bs%d_zp%d" % s)
def test_f32_rows_at_a_level_that_allows_f16_activations(ctx, pkg, oracle, shape, level, options):
    """accuracy_level 2, 3 and 4 allow the activations to be reduced to f16, bf16 or int8 (the reference never reads
    the attribute and computes in f32). More than 32 rows of f32 then travel as ONE f16 row each: the row times the
    power of two that puts its largest value into [2^14, 2^15), rounded to f16 (11 bits of every value, whatever the
    row's size). The result is the operator on exactly those rounded rows, at the f32 tolerance -- and so within
    what each of the three levels permits."""
    m, k, n, bs, with_zp = shape
    B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=45, with_zp=with_zp)
    a = pkg.synth.normal_f32(m * k, 46).reshape(m, k)
    a[0] *= np.float32(3.0e7)
    a[1] *= np.float32(1.0e-9)
    a[2] = 0
    mx = np.abs(a).max(axis=1, keepdims=True)
    e = np.where(mx > 0, np.floor(np.log2(np.maximum(mx, np.float32(1e-30)))) - 14, 0).astype(np.int32)
    rounded = np.ldexp(np.ldexp(a, -e).astype(np.float16).astype(np.float32), e).astype(np.float32)
    assert np.all(np.abs(rounded - a) <= 2.0 ** -11 * mx)
    want = oracle.matmul_nbits(rounded, B, scales, zp, k, n, bs)
    w = pkg.ops.NBitsWeight(ctx, B, scales, zp, k, n, bs)
    with ctx.options(**options):
        got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, accuracy_level=level, weight=w)
    w.destroy()
    assert got.dtype == np.float32 and got.shape == (m, n)
    scale = np.maximum(np.abs(want).max(axis=1, keepdims=True), 1e-30)
    assert np.all(np.abs(got - want) <= (1e-3 + 1e-4 * np.abs(want)) * np.maximum(scale / np.abs(want[3:]).max(), 1e-30) + 1e-4 * scale), worst(got, want)
    assert np.all(got[2] == 0)


@pytest.mark.parametrize("options", [{}, {"HIPC_PREFILL_TILE": 128, "HIPC_PREFILL_SPLIT": 2}, {"HIPC_PREFILL_TILE": 192}, {"HIPC_PREFILL_DIRECT": 0}],
                         ids=lambda v: str(v).replace(" ", ""))
@pytest.mark.parametrize("shape", F32_PREFILL, ids=lambda s: "M%d_K%d_N%d_bs%d_zp%d" % s)
def test_f32_rows_with_f32_pinned(ctx, pkg, oracle, shape, options):
    """accuracy_level 1 pins f32: more than 32 rows travel as THREE f16 rows each (every bit of the row's values
    beside its power of two) through the tiled kernel, and a launch adds the three results. Against the oracle at
    the operator's tolerance; against the float64 product no worse than the default's two terms, and within what f32
    accumulation leaves."""
    m, k, n, bs, with_zp = shape
    B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=45, with_zp=with_zp)
    a = pkg.synth.normal_f32(m * k, 46).reshape(m, k)
    a[0] *= np.float32(3.0e7)
    a[1] *= np.float32(1.0e-9)
    a[2] = 0
    want = oracle.matmul_nbits(a, B, scales, zp, k, n, bs)
    w = pkg.ops.NBitsWeight(ctx, B, scales, zp, k, n, bs)
    with ctx.options(**options):
        got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, accuracy_level=1, weight=w)
        two = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, weight=w)
    w.destroy()
    scale = np.maximum(np.abs(want).max(axis=1, keepdims=True), 1e-30)
    assert np.all(np.abs(got - want) <= (1e-3 + 1e-4 * np.abs(want)) * np.maximum(scale / np.abs(want[3:]).max(), 1e-30) + 1e-4 * scale), worst(got, want)
    nib, z = _unpack(B, zp if zp is not None else np.full((n, (-(-k // bs) + 1) // 2), 0x88, np.uint8), k, n, bs)
    f64 = rc.matmul_nbits_f64(a, nib, z, scales.reshape(n, -1), bs)
    big = np.maximum(np.abs(f64).max(axis=1, keepdims=True), 1e-300)
    e3, e2 = np.abs(got - f64) / big, np.abs(two - f64) / big
    assert e3.max() <= 2e-5, float(e3.max())
    assert e3.max() <= e2.max() * 1.05 + 1e-7, (float(e3.max()), float(e2.max()))
    assert np.all(got[2] == 0)


@pytest.mark.parametrize("groups", [1, 2])
@pytest.mark.parametrize("tile", [64, 128, 192])
@pytest.mark.parametrize("level", [0, 1])
@pytest.mark.parametrize("shape", [(33, 70, 70, 32, True), (64, 128, 128, 32, False), (65, 448, 129, 64, True), (97, 1100, 257, 128, False), (129, 576, 300, 256, True)],
                         ids=lambda s: "M%d_K%d_N%d_bs%d_zp%d" % s)
def test_terms_of_f32_rows_added_in_one_accumulator(ctx, pkg, shape, level, tile, groups):
    """Every tile that holds the two (level 1: three) f16 terms of its f32 rows in one wavefront, with one k group per workgroup
    and with several: rows and columns one past a tile, fewer stages than groups, a partial last stage. Against float64:
    what the terms leave of a row's largest value times the column's absolute sum, and f32 accumulation over k."""
    m, k, n, bs, with_zp = shape
    B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=47, with_zp=with_zp)
    a = pkg.synth.normal_f32(m * k, 48).reshape(m, k)
    a[m - 1] *= np.float32(1.0e7)
    nib, z = _unpack(B, zp if zp is not None else np.full((n, (-(-k // bs) + 1) // 2), 0x88, np.uint8), k, n, bs)
    f64 = rc.matmul_nbits_f64(a, nib, z, scales.reshape(n, -1), bs)
    absw = rc.matmul_nbits_f64(np.ones((1, k)), np.abs(nib.astype(np.int64) - z.repeat(bs, axis=1)[:, :k]), np.zeros_like(z), scales.reshape(n, -1), bs)
    absy = rc.matmul_nbits_f64(np.abs(a), np.abs(nib.astype(np.int64) - z.repeat(bs, axis=1)[:, :k]), np.zeros_like(z), scales.reshape(n, -1), bs)
    bound = np.abs(a).max(axis=1, keepdims=True).astype(np.float64) * 2.0 ** (-24 if level else -21) * absw + (k + 8) * 2.0 ** -24 * absy
    w = pkg.ops.NBitsWeight(ctx, B, scales, zp, k, n, bs)
    with ctx.options(HIPC_PREFILL_TILE=tile, HIPC_PREFILL_GROUPS=groups):
        got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, accuracy_level=level, weight=w)
    w.destroy()
    assert got.dtype == np.float32 and got.shape == (m, n)
    assert np.all(np.abs(got - f64) <= bound), float(np.max(np.abs(got - f64) / bound))


@pytest.mark.parametrize("shape", [(400, 192, 1152, 32, True), (400, 136, 1090, 64, False), (384, 192, 1024, 128, True)], ids=lambda s: "M%d_K%d_N%d_bs%d_zp%d" % s)
def test_f32_rows_by_the_tiles_an_xcd_gets(ctx, pkg, shape):
    """Two terms on either side of the rule that leaves 64x64 tiles where one XCD would get more of them than it has CUs (35, 35
    and 32 of 32): against float64, within the bound of the test above."""
    m, k, n, bs, with_zp = shape
    B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=67, with_zp=with_zp)
    a = pkg.synth.normal_f32(m * k, 68).reshape(m, k)
    nib, z = _unpack(B, zp if zp is not None else np.full((n, (-(-k // bs) + 1) // 2), 0x88, np.uint8), k, n, bs)
    w64 = (nib.astype(np.float64) - z.repeat(bs, axis=1)[:, :k]) * scales.reshape(n, -1).astype(np.float64).repeat(bs, axis=1)[:, :k]
    absw = np.abs(w64)
    bound = np.abs(a).max(axis=1, keepdims=True).astype(np.float64) * 2.0 ** -21 * absw.sum(axis=1) + (k + 8) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ absw.T)
    got = pkg.ops.matmul_nbits(ctx, a, B, scales, zp, k, n, bs)
    err = np.abs(got - a.astype(np.float64) @ w64.T)
    assert np.all(err <= bound), float(np.max(err / bound))


@pytest.mark.parametrize("shape", [(33, 1152, 64, 32, True), (64, 1096, 1154, 64, False), (100, 2056, 257, 128, True), (200, 4096, 130, 32, False),
                                   (400, 1152, 1152, 128, True), (1000, 776, 1030, 256, False)], ids=lambda s: "M%d_K%d_N%d_bs%d_zp%d" % s)
def test_f32_pinned_rows_with_k_split_by_shape(ctx, pkg, shape):
    """Three terms where the estimate picks the tile and splits k two to four ways, with one group of wavefronts and several, a
    partial last stage, columns one past a tile: against float64, within the bound of the test above."""
    m, k, n, bs, with_zp = shape
    B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=57, with_zp=with_zp)
    a = pkg.synth.normal_f32(m * k, 58).reshape(m, k)
    a[m // 2] *= np.float32(1.0e-6)
    nib, z = _unpack(B, zp if zp is not None else np.full((n, (-(-k // bs) + 1) // 2), 0x88, np.uint8), k, n, bs)
    w64 = (nib.astype(np.float64) - z.repeat(bs, axis=1)[:, :k]) * scales.reshape(n, -1).astype(np.float64).repeat(bs, axis=1)[:, :k]
    absw = np.abs(w64)
    bound = np.abs(a).max(axis=1, keepdims=True).astype(np.float64) * 2.0 ** -24 * absw.sum(axis=1) + (k + 8) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ absw.T)
    w = pkg.ops.NBitsWeight(ctx, B, scales, zp, k, n, bs)
    for options in ({}, {"HIPC_PREFILL_SPLIT": 0}):
        with ctx.options(**options):
            got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, accuracy_level=1, weight=w)
        err = np.abs(got - a.astype(np.float64) @ w64.T)
        assert np.all(err <= bound), float(np.max(err / bound))
    w.destroy()


@pytest.mark.parametrize("kn", [(2048, 11008), (11008, 2048), (2048, 2560)], ids=lambda s: "K%d_N%d" % s)
def test_prefill_configuration_full_size(ctx, pkg, oracle, kn):
    """512 rows of f16 activations against block-128 symmetric weights with f16 scales (no zero
    points: 8 is implied), the three linears of the prefill configuration at full size."""
    k, n = kn
    m, bs = 512, 128
    B, scales, _ = pkg.synth.fast_nbits_weight(n, k, bs, seed=43, with_zp=False, scale_dtype=np.float16)
    a = pkg.synth.normal_f32(m * k, 44).reshape(m, k).astype(np.float16)
    want = oracle.matmul_nbits(a, B, scales, None, k, n, bs)
    w = pkg.ops.NBitsWeight(ctx, B, scales, None, k, n, bs)
    got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, weight=w)
    # linearity in A, a size-independent property: f(2a) == 2 f(a) exactly (a power of two scales every product, every
    # partial sum and the rounding to a normal f16 alike)
    got2 = pkg.ops.matmul_nbits(ctx, (2 * a).astype(np.float16), None, None, None, k, n, bs, weight=w)
    w.destroy()
    assert close(got, want, RTOL16), worst(got, want)
    normal = np.abs(got.astype(np.float32)) >= 2.0 ** -13   # (a subnormal f16 result has no spare bit to double into)
    assert np.array_equal(got2.astype(np.float32)[normal], 2 * got.astype(np.float32)[normal]) and normal.mean() > 0.99


def test_unembedding_width_full_size(ctx, pkg, oracle):
    """lm_head of the decoder configuration: K = 1152, N = 262144, every column checked."""
    k, n, bs = 1152, 262144, 32
    B, scales, zp = pkg.synth.fast_nbits_weight(n, k, bs, seed=17)
    a = pkg.synth.normal_f32(k, 18).reshape(1, k)
    want = oracle.matmul_nbits(a, B, scales, zp, k, n, bs)
    w = pkg.ops.NBitsWeight(ctx, B, scales, zp, k, n, bs)
    got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, weight=w)
    assert close(got, want, RTOL32), worst(got, want)
    # linearity in A, a size-independent property: f(2a) == 2 f(a) exactly (power-of-two scaling)
    got2 = pkg.ops.matmul_nbits(ctx, 2 * a, None, None, None, k, n, bs, weight=w)
    assert np.array_equal(got2, 2 * got)
    w.destroy()


def test_refusals_and_short_buffers(ctx, pkg):
    k, n, bs = 128, 16, 32
    B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=1)
    a = np.zeros((1, k), np.float32)
    with pytest.raises(pkg.HipComputeError) as e:   # the operator defines levels 0..4
        pkg.ops.matmul_nbits(ctx, a, B, scales, zp, k, n, bs, accuracy_level=5)
    assert e.value.code == 2
    with pytest.raises(pkg.HipComputeError) as e:   # the weight is short for N (interp.rs:6465-6472)
        pkg.ops.matmul_nbits(ctx, a, B[: n - 1], scales, zp, k, n, bs)
    assert e.value.code == 1 and "short" in e.value.message
    with pytest.raises(pkg.HipComputeError) as e:   # not a multiple of 8: a packed word would straddle two blocks
        pkg.ops.matmul_nbits(ctx, a, B, scales, zp, k, n, 20)
    assert e.value.code == 1
    y = pkg.ops.matmul_nbits(ctx, np.zeros((0, k), np.float32), B, scales, zp, k, n, bs)   # no rows: a no-op
    assert y.shape == (0, n)


def _unpack(B, zp, k, n, bs):
    nb = -(-k // bs)
    flat = B.reshape(n, -1)
    nib = np.empty((n, nb * bs), np.uint8)
    nib[:, 0::2], nib[:, 1::2] = flat & 15, flat >> 4
    z = np.empty((n, 2 * zp.shape[1]), np.uint8)
    z[:, 0::2], z[:, 1::2] = zp & 15, zp >> 4
    return nib[:, :k], z[:, :nb]


@pytest.mark.parametrize("shape", [(1, 1152, 6912), (1, 6912, 1152), (8, 1152, 512), (1, 1152, 32768 + 48)], ids=lambda s: "M%d_K%d_N%d" % s)
def test_accuracy_levels(ctx, pkg, oracle, shape):
    """accuracy_level 0 (unset), 2, 3 and 4 (a lower bound: the reference computes every level in f32) let
    an f32 activation enter the matrix cores as two bf16 terms; 1 pins f32 and sends all 24 bits (three terms). The last shape has more than 2048 column tiles, so
    its one row takes the wide streaming kernel (the unembedding's route) and level 1 that kernel's
    three-term instance. Every level meets the operator's tolerance
    against the oracle; level 1 is held to a tighter bound against the float64 product -- 2e-5 of
    the row's largest output, what the f32 accumulation of the +128-biased block dots leaves --
    and must not be worse than the default."""
    m, k, n = shape
    bs = 32
    B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=300 + n)
    a = pkg.synth.normal_f32(m * k, 301).reshape(m, k)
    want = oracle.matmul_nbits(a, B, scales, zp, k, n, bs)
    nib, z = _unpack(B, zp, k, n, bs)
    f64 = rc.matmul_nbits_f64(a, nib, z, scales.reshape(n, -1), bs)
    w = pkg.ops.NBitsWeight(ctx, B, scales, zp, k, n, bs)
    err = {}
    for level in (0, 1, 2, 3, 4):
        got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, accuracy_level=level, weight=w)
        assert close(got, want, RTOL32), (level, worst(got, want))
        err[level] = float(np.max(np.abs(got - f64)))
    w.destroy()
    assert err[1] <= 2e-5 * float(np.max(np.abs(f64))), err
    assert err[1] <= err[0] * 1.05 + 1e-7, err
    assert err[2] == err[0] and err[3] == err[0] and err[4] == err[0], err     # the same kernel instance as the default


@pytest.mark.parametrize("shape", [(1, 1152, 6912, 32, True), (1, 6912, 1152, 32, True), (1, 2048, 2560, 128, False),
                                   (1, 300, 100, 64, True), (1, 1024, 48, 32, True)], ids=lambda s: "M%d_K%d_N%d_bs%d_zp%d" % s)
def test_one_row_on_the_streaming_kernel(ctx, pkg, oracle, shape):
    """One f32 row takes the kernel built for latency by default; with the HIPC_GEMV_LEAN option at 0 the
    same product runs on the streaming kernel: both against the oracle, and against each other."""
    m, k, n, bs, with_zp = shape
    B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=400 + n, with_zp=with_zp)
    a = pkg.synth.normal_f32(m * k, 401).reshape(m, k)
    want = oracle.matmul_nbits(a, B, scales, zp, k, n, bs)
    w = pkg.ops.NBitsWeight(ctx, B, scales, zp, k, n, bs)
    lean = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, weight=w)
    with ctx.options(HIPC_GEMV_LEAN=0):
        streaming = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, weight=w)
    w.destroy()
    assert close(lean, want, RTOL32), ("lean", worst(lean, want))
    assert close(streaming, want, RTOL32), ("streaming", worst(streaming, want))
    assert close(lean, streaming, RTOL32)


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("bs,with_zp", [(32, True), (64, False), (128, True)])
@pytest.mark.parametrize("shape", [(2, 136, 40), (4, 1152, 1030), (5, 1000, 200), (8, 2056, 16), (9, 72, 600), (16, 4096, 272), (17, 1288, 90),
                                   (32, 520, 1040), (33, 2048, 131), (64, 1152, 96), (64, 264, 2064), (7, 8, 33)], ids=lambda s: "M%d_K%d_N%d" % s)
def test_a_few_rows(ctx, pkg, oracle, shape, bs, with_zp, dtype):
    """2 to 64 rows: every number of row blocks and result registers, rows that fill their stage of LDS once and several
    times, k split over workgroups, a last tile of k with eight values, columns that end inside a tile."""
    m, k, n = shape
    B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=500 + n, with_zp=with_zp, scale_dtype=dtype)
    a = pkg.synth.normal_f32(m * k, 501).reshape(m, k).astype(dtype)
    w = pkg.ops.NBitsWeight(ctx, B, scales, zp, k, n, bs)
    want = oracle.matmul_nbits(a, B, scales, zp, k, n, bs)
    got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, weight=w)
    assert close(got, want, RTOL32 if dtype == np.float32 else RTOL16), worst(got, want)
    w.destroy()


@pytest.mark.parametrize("m", [3, 16, 20])
@pytest.mark.parametrize("level", [0, 1])
def test_a_few_rows_of_very_different_size(ctx, pkg, oracle, m, level):
    """Rows that are not split as they are: values above 2^15, rows whose largest value is small, subnormal, zero."""
    k, n, bs = 640, 80, 32
    B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=511)
    a = pkg.synth.normal_f32(m * k, 512).reshape(m, k)
    a[0] *= np.float32(1e30)
    a[1] *= np.float32(1e-20)
    a[2] = 0
    a[m - 1, ::3] *= np.float32(1e5)
    w = pkg.ops.NBitsWeight(ctx, B, scales, zp, k, n, bs)
    want = oracle.matmul_nbits(a.astype(np.float32), B, scales, zp, k, n, bs)
    got = pkg.ops.matmul_nbits(ctx, a.astype(np.float32), None, None, None, k, n, bs, accuracy_level=level, weight=w)
    for r in range(m):   # each row against its own size
        assert np.max(np.abs(got[r] - want[r])) <= 1e-5 * max(np.max(np.abs(want[r])), 1e-37), r
    w.destroy()


@pytest.mark.parametrize("dtype,level", [(np.float16, 0), (np.float32, 0), (np.float32, 4)])
@pytest.mark.parametrize("shape", [(1, 1160, 1030), (2, 512, 1040), (16, 2056, 200), (20, 136, 600), (43, 1288, 96), (65, 1000, 131), (130, 648, 400), (300, 1152, 1100)],
                         ids=lambda s: "M%d_K%d_N%d" % s)
def test_blocks_of_sixteen_on_the_matrix_cores(ctx, pkg, oracle, shape, dtype, level):
    """Blocks of 16, two to a product step of the kernel for a few rows, one to a step of the tiled kernel (64- and
    128-row tiles): a last block with eight values, an odd number of blocks, rows that do not start on 16 bytes."""
    m, k, n = shape
    B, scales, zp = pkg.synth.nbits_weight(n, k, 16, seed=600 + n, scale_dtype=dtype)
    a = pkg.synth.normal_f32(m * k, 601).reshape(m, k).astype(dtype)
    w = pkg.ops.NBitsWeight(ctx, B, scales, zp, k, n, 16)
    want = oracle.matmul_nbits(a, B, scales, zp, k, n, 16)
    got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, 16, accuracy_level=level, weight=w)
    assert got.dtype == dtype
    if level:    # one f16 term of a row from 33 rows on: 11 bits of every value
        assert worst(got, want) <= 1e-3 * np.abs(want).max()
    else:
        assert close(got, want, RTOL16 if dtype == np.float16 else RTOL32), worst(got, want)
    moved = ctx.upload(np.concatenate([np.zeros(2, dtype), a.reshape(-1)]))
    out = ctx.alloc(m * n * a.itemsize)
    pkg.ops.matmul_nbits_packed_device(ctx, moved.at(2 * a.itemsize), pkg.ops.hipc_dtype(a.dtype), w, out, m, level)
    assert np.array_equal(ctx.download(out, dtype, (m, n)), got)
    moved.free(), out.free(), w.destroy()


@pytest.mark.parametrize("bs,level", [(16, 0), (32, 0), (64, 0), (128, 0), (32, 4)])
@pytest.mark.parametrize("shape", [(65, 1024, 130), (95, 520, 64), (97, 1160, 1100), (128, 648, 96), (70, 4224, 200), (66, 8200, 100)], ids=lambda s: "M%d_K%d_N%d" % s)
def test_f32_rows_on_small_tiles(ctx, pkg, oracle, shape, bs, level):
    """Rows of f32 on 64-row tiles: the last tile with one row, one missing and full; one group of wavefronts and two;
    k split over workgroups (k of 4224 and more), the last split shorter than the others."""
    m, k, n = shape
    B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=700 + n)
    a = pkg.synth.normal_f32(m * k, 701).reshape(m, k)
    a[0] *= np.float32(1e20)
    w = pkg.ops.NBitsWeight(ctx, B, scales, zp, k, n, bs)
    want = oracle.matmul_nbits(a, B, scales, zp, k, n, bs)
    got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, accuracy_level=level, weight=w)
    for rows in (slice(0, 1), slice(1, m)):   # the large row against its own size
        assert np.max(np.abs(got[rows] - want[rows])) <= (1e-3 if level else 1e-5) * np.max(np.abs(want[rows])), rows
    w.destroy()


def unpacked(B, scales, zp, k, n, bs):
    """The weight's (q - zp) and scales, [N, K] in 64 bits."""
    nb = -(-k // bs)
    codes = np.stack([B & 15, B >> 4], axis=-1).reshape(n, -1)[:, :k].astype(np.float64)
    if zp is None:
        z = np.full((n, nb), 8.0)
    else:
        z = np.stack([zp & 15, zp >> 4], axis=-1).reshape(n, -1)[:, :nb].astype(np.float64)
    s = np.asarray(scales).reshape(n, nb).astype(np.float64)
    return codes - np.repeat(z, bs, axis=1)[:, :k], np.repeat(s, bs, axis=1)[:, :k]


@pytest.mark.parametrize("bs", [16, 32, 128])
@pytest.mark.parametrize("level", [0, 1])
@pytest.mark.parametrize("m", [1, 3, 16, 20, 40, 70])
def test_rows_of_tiny_values(ctx, pkg, oracle, m, level, bs):
    """Rows whose largest value lies anywhere down to the smallest normal number, subnormal rows, and an ordinary row
    with a run of tiny values (a whole slice of k, where k is split over workgroups): the power of two a row is scaled by
    stays a number. Scales near 2^10 keep the results in the normal range, so the bound is the rows' own."""
    k, n = 2176, 80
    B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=521)
    scales = (scales * np.float32(2.0**15)).astype(np.float32)
    a = pkg.synth.normal_f32(m * k, 522).reshape(m, k)
    a /= np.abs(a).max(axis=1, keepdims=True)           # the largest of a row is 1
    for r in range(m):
        a[r] *= np.float32(2.0) ** -(110 + (7 * r + 3) % 18)      # 2^-110 .. 2^-127
    a[m // 2] = pkg.synth.normal_f32(k, 523)
    a[m // 2, 128:1280] *= np.float32(2.0**-113)
    w = pkg.ops.NBitsWeight(ctx, B, scales, zp, k, n, bs)
    got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, accuracy_level=level, weight=w)
    w.destroy()
    d, s = unpacked(B, scales, zp, k, n, bs)
    want = a.astype(np.float64) @ (d * s).T
    assert np.all(np.isfinite(got))
    for r in range(m):
        # 16 bits of a value or better (2^-16, over sqrt(K) of them), an f32 sum, and subnormal inputs' own last bits
        assert np.max(np.abs(got[r] - want[r])) <= 2e-5 * np.max(np.abs(want[r])) + 2.0**-149 * np.sum(np.abs(d * s), axis=1).max(), r


@pytest.mark.parametrize("m", [2, 8, 16, 24, 40])
@pytest.mark.parametrize("bs,level", [(32, 0), (64, 1), (128, 0), (16, 0), (16, 1)])
def test_small_values_beside_a_large_one(ctx, pkg, bs, level, m):
    """An activation row as language models have them, one value of ordinary size among small ones, against columns whose
    weight for that value is zero: the small ones count in full. They are whole multiples of 2^-32 times at most 127, so
    every sum is exact in f32 and so must the result be: two f16 terms of a scaled row hold any 22 bits that end 2^-31 below
    a largest value near 1 or earlier."""
    k, n = 640, 48
    rng = np.random.default_rng(77)
    q = np.full((n, k), 8, np.uint8)
    small = rng.choice(np.arange(1, k), 32, replace=False)
    q[:, small] = rng.integers(0, 16, (n, 32))
    B = pkg.synth.pack_nibbles(q, bs)
    scales = np.ones(n * (-(-k // bs)), np.float32)
    a = np.zeros((m, k), np.float32)
    a[:, 0] = 0.6
    a[:, small] = rng.integers(-127, 128, (m, 32)) * 2.0**-32
    w = pkg.ops.NBitsWeight(ctx, B, scales, None, k, n, bs)
    got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, accuracy_level=level, weight=w)
    w.destroy()
    want = a[:, small].astype(np.float64) @ (q[:, small].astype(np.float64) - 8).T
    assert np.array_equal(got, want.astype(np.float32))


@pytest.mark.parametrize("m", [1, 2, 16, 20, 40, 70])
@pytest.mark.parametrize("bs,level", [(16, 0), (16, 1), (32, 1)])
def test_every_bit_of_a_small_value_beside_a_large_one(ctx, pkg, bs, level, m):
    """Where three terms are promised (accuracy_level 1, and blocks of 16, unless a level allows less): 24 significant
    bits of a value 2^30 times smaller than the row's largest. One product per result, so the result is that product,
    correctly rounded but for the bias some kernels carry (the nearest f32, or its neighbours)."""
    k, n = 512, 32
    rng = np.random.default_rng(78)
    q = np.full((n, k), 8, np.uint8)
    q[:, 7] = rng.integers(9, 16, n)
    B = pkg.synth.pack_nibbles(q, bs)
    scales = np.ones(n * (k // bs), np.float32)
    a = np.zeros((m, k), np.float32)
    a[:, 300] = 1.5
    a[:, 7] = (rng.integers(1 << 23, 1 << 24, m) | 1) * 2.0**-53
    w = pkg.ops.NBitsWeight(ctx, B, scales, None, k, n, bs)
    got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, accuracy_level=level, weight=w)
    w.destroy()
    want = np.outer(a[:, 7].astype(np.float64), q[:, 7].astype(np.float64) - 8)
    # the terms leave up to half a unit of the value's last bit, and f32 rounds the product and the terms' sum once each;
    # one row of blocks of 32 is multiplied as 128 + q, and 128 + zp taken back: roundings at 143 times the result's size
    bound = 4 * 2.0**-24 * (143 if m == 1 and bs == 32 else 1)
    assert np.all(np.abs(got - want) <= bound * np.abs(want))


@pytest.mark.parametrize("dtype", [np.float32, np.float16])
@pytest.mark.parametrize("m", [1, 3, 16, 20, 40, 70])
def test_infinite_activations_with_blocks_of_sixteen(ctx, pkg, m, dtype):
    """One infinite value in a row: what the operator's own layout gives -- an infinity of the product's sign, NaN where
    the weight is zero -- and nothing in other rows."""
    k, n, bs = 512, 64, 16
    B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=531, scale_dtype=dtype)
    a = pkg.synth.normal_f32(m * k, 532).reshape(m, k).astype(dtype)
    a[0, 37] = np.inf
    if m > 2:
        a[2, 500] = -np.inf
        a[1, 3] = 6e4 if dtype == np.float16 else 1e8       # (finite)
    want = pkg.ops.matmul_nbits(ctx, a[:, :], B, scales, zp, k, n, bs) if m <= 16 else None
    d, s = unpacked(B, scales, zp, k, n, bs)
    w = pkg.ops.NBitsWeight(ctx, B, scales, zp, k, n, bs)
    got = pkg.ops.matmul_nbits(ctx, a, None, None, None, k, n, bs, weight=w)
    w.destroy()
    for r, at, sign in ((0, 37, 1), (2, 500, -1)):
        if r >= m:
            continue
        zero = d[:, at] == 0
        assert np.all(np.isnan(got[r][zero])) and np.array_equal(got[r][~zero], sign * np.sign(d[~zero, at]) * np.inf)
        assert want is None or np.array_equal(got[r], want[r], equal_nan=True)
    rest = [r for r in range(m) if r not in (0, 2)]
    exact = a[rest].astype(np.float64) @ (d * s).T
    with np.errstate(over="ignore"):
        assert np.all(np.isfinite(got[rest]) == np.isfinite(exact.astype(dtype)))
    ok = np.isfinite(got[rest])
    assert np.all(np.abs(got[rest] - exact)[ok] <= (1e-2 if dtype == np.float16 else 1e-3) + 2e-3 * np.abs(exact)[ok])


FIRST_IN_A_CAPTURE = [  # (M, K, N, block, activations, elements the rows are off 16 bytes): what an unrecorded first call wants scratch memory for
    (2, 4096, 256, 32, np.float32, 0),       # k split over workgroups
    (6, 6912, 1152, 128, np.float16, 0),
    (24, 640, 600, 32, np.float32, 0),       # rows split into terms by a launch in front
    (100, 8192, 1024, 64, np.float16, 0),    # 64-row tiles with k split
    (1, 6912, 1152, 16, np.float32, 0), (16, 4096, 272, 16, np.float32, 0), (20, 1288, 600, 16, np.float32, 0), (65, 1000, 131, 16, np.float32, 0),
    (100, 8192, 1024, 16, np.float16, 0),
    (1, 1160, 130, 16, np.float32, 1), (5, 1160, 130, 16, np.float16, 1), (43, 520, 96, 16, np.float32, 2),   # rows off 16 bytes
]


@pytest.mark.parametrize("layout", ["handle", "operator"])
@pytest.mark.parametrize("case", FIRST_IN_A_CAPTURE, ids=lambda c: "M%d_K%d_N%d_bs%d_%s_off%d" % (*c[:4], c[4].__name__, c[5]))
def test_a_first_call_inside_a_capture(pkg, oracle, case, layout):
    """A context that has never run the operator records it: scratch memory cannot grow there, and the call takes a route
    that needs none, or is refused. The graph is replayed with eager work in between, which may then grow the scratch memory."""
    m, k, n, bs, dtype, off = case
    refused = layout == "operator" and bs != 16 and m > (32 if dtype == np.float32 else 16)   # the tiled form would go to scratch memory
    B, scales, zp = pkg.synth.nbits_weight(n, k, bs, seed=541, scale_dtype=dtype)
    a = pkg.synth.normal_f32(m * k, 542).reshape(m, k).astype(dtype)
    want = oracle.matmul_nbits(a, B, scales, zp, k, n, bs)
    rtol = RTOL32 if dtype == np.float32 else RTOL16
    with pkg.Context(0) as c:
        dt = pkg.ops.hipc_dtype(a.dtype)
        dA = c.upload(np.concatenate([np.zeros(off, dtype), a.reshape(-1)]))
        dY = c.alloc(m * n * a.itemsize)
        if layout == "handle":
            w = pkg.ops.NBitsWeight(c, B, scales, zp, k, n, bs)
            call = lambda: pkg.ops.matmul_nbits_packed_device(c, dA.at(off * a.itemsize), dt, w, dY, m)  # noqa: E731
        else:
            held = [c.upload(v) for v in (B, scales, zp)]
            call = lambda: pkg.ops.matmul_nbits_device(c, dA.at(off * a.itemsize), dt, held[0], B.size, held[1], dt, scales.size, held[2], zp.size, dY, m, k, n, bs)  # noqa: E731
        c.flush()
        c.capture_begin()
        try:
            if refused:
                with pytest.raises(pkg.HipComputeError) as e:
                    call()
                assert e.value.code == 2
            else:
                call()
        finally:
            graph = c.capture_end()
        for _ in range(0 if refused else 3):
            c.fill(dY, 0, m * n * a.itemsize // 4 * 4, 0)
            c.graph_launch(graph)
            got = c.download(dY, dtype, (m, n))
            assert close(got, want, rtol), worst(got, want)
            call()
            assert close(c.download(dY, dtype, (m, n)), want, rtol)
        c.graph_destroy(graph)
        if layout == "handle":
            w.destroy()


def test_a_weight_in_blocks_of_sixteen_beyond_the_tiled_form(ctx, pkg):
    """4 GiB of nibbles: more than the tiled form's 32-bit offsets reach, so the handle keeps the operator's layout. Codes
    10 and 5 under zero point 8, scale 1, activations 1: each result is (2 - 3) K / 2."""
    k, n, bs = 4096, 1 << 21, 16
    blocks = k // bs
    b_len = n * blocks * (bs // 2)
    B, S = ctx.alloc(b_len), ctx.alloc(n * blocks * 4)
    ctx.fill(B, 0, b_len, 0x5A5A5A5A)
    ctx.fill(S, 0, n * blocks * 4, 0x3F800000)
    import ctypes as C
    h = C.c_void_p()
    ctx._check(ctx.lib.hipc_prepack_matmul_nbits(ctx.handle, B.ptr, b_len, S.ptr, pkg.F32, n * blocks, None, 0, k, n, bs, C.byref(h)))
    B.free(), S.free()
    assert ctx.lib.hipc_nbits_weight_bytes(h) == b_len + n * blocks * 4
    dA = ctx.upload(np.ones(k, np.float32))
    dY = ctx.alloc(n * 4)
    ctx._check(ctx.lib.hipc_matmul_nbits_packed(ctx.handle, dA.ptr, pkg.F32, h, dY.ptr, 1, 0))
    got = ctx.download(dY, np.float32, (n,))
    ctx.lib.hipc_nbits_weight_destroy(ctx.handle, h)
    dA.free(), dY.free()
    ctx.flush()
    assert np.all(got == -k / 2)
