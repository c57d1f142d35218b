"""The prompt GEMM's block shapes (gemm.hip: 32 or 64 rows by 128, 64 or 32
outputs, the sum whole or in 2 or 4 parts) and the rule that takes them, at
their edges: one row and output past a tile, sums of one group, of a part of
a chunk and of chunks that leave waves idle, rows around the 8-row launches'
limit, against the CPU oracle's Linear.

Bound: the group sums are exact integers and the scales multiply in double, so
only the order of a double sum differs from the CPU's: a value differs by at
most one ulp of single, in at most 1/1000 of the values (the bound of the
other Linear tests)."""
import numpy as np
import pytest

import infer_hip as H
import oracle_lib as O

pytestmark = pytest.mark.gpu

BLOCK = [H.Q8_0, H.Q4_0, H.MXFP4, H.Q5_0, H.Q5_1, H.Q4_K, H.Q6_K]
# (rows, in, out): four shapes of tiles, the edges of the rule between them
SHAPES = [(9, 32, 6144), (9, 256, 3073), (12, 288, 3200), (17, 2048, 2100), (33, 1056, 1025),
          (80, 512, 33), (81, 3328, 129), (97, 1280, 8193), (257, 768, 4100), (1024, 256, 2049),
          (1023, 544, 4097)]


@pytest.fixture(scope="module")
def ctx():
    c = H.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("dtype", BLOCK, ids=[H.NAMES[t] for t in BLOCK])
def test_tiles_match_oracle(ctx, dtype):
    for rows, cols, out in SHAPES:
        if cols % H.BLOCK[dtype][0]:
            cols = -(-cols // 256) * 256
        rng = np.random.default_rng(rows + out)
        x = rng.standard_normal((rows, cols)).astype(np.float32)
        x[:, ::61] *= 9
        x[rows // 2] = 0
        bias = rng.standard_normal(out).astype(np.float32)
        w = H.synth_blocks(dtype, out, cols, rows + cols, -8, -4)
        got = ctx.linear(x, w, dtype, out, bias, mode=H.MODE_Q8)
        ref = O.linear(x, w, dtype, out, bias)
        bits = np.abs(got.view(np.int32).astype(np.int64) - ref.view(np.int32).astype(np.int64))
        print(H.NAMES[dtype], rows, cols, out, "differ", int((bits > 0).sum()), flush=True)
        # (a value within a rounding of zero may change its sign bit: compared by size)
        near = np.abs(got - ref) <= np.abs(ref) * 2.0 ** -23 + 1e-30
        assert np.all((bits <= 1) | near), (rows, cols, out, int(bits.max()))
        assert (bits > 0).mean() <= 1e-3


def same(got, ref):
    """At most one ulp of single apart, in at most 1/1000 of the values."""
    bits = np.abs(got.view(np.int32).astype(np.int64) - ref.view(np.int32).astype(np.int64))
    # (a value within a rounding of zero may change its sign bit: compared by size)
    near = np.abs(got - ref) <= np.abs(ref) * 2.0 ** -23 + 1e-30
    assert np.all((bits <= 1) | near), int(bits.max())
    assert (bits > 0).mean() <= 1e-3


# (rows, in, out, the parts of the sum on 256 CUs): by the 32 x 128 tiles and
# the sum's chunks of 256 values, no part without a chunk
PARTS = [(80, 256, 6144, 1), (97, 256, 130, 1), (300, 512, 2048, 2), (100, 512, 700, 2), (200, 768, 700, 4),
         (200, 768, 3072, 2), (200, 768, 3500, 1), (300, 1024, 2048, 2), (300, 1280, 2048, 2),
         (300, 1536, 2048, 4), (300, 2048, 1024, 4), (200, 2048, 3500, 2), (520, 1024, 4000, 1)]


@pytest.mark.parametrize("rows,cols,out,parts", PARTS)
def test_parts_of_the_sum(ctx, rows, cols, out, parts):
    if ctx.info()[2] != 256:
        pytest.skip("the line lies at other sizes on another number of CUs")
    x = np.random.default_rng(rows + out).standard_normal((rows, cols)).astype(np.float32)
    for dtype in (H.Q4_0, H.Q6_K):
        w = H.synth_blocks(dtype, out, cols, rows + cols, -8, -4)
        ctx.kernel_timer("gemm", 16)
        got = ctx.linear(x, w, dtype, out, mode=H.MODE_Q8)
        names = list(ctx.kernel_timer_report())
        ctx.kernel_timer(None)
        assert names == ["gemm_%s_m1k%d" % (H.NAMES[dtype].lower(), parts)]
        same(got, O.linear(x, w, dtype, out, None))


# (type, rows, in, out, on the GEMM): 9 to 79 rows on either side of the line
# to the 8-row launches, which depends on the type and on how those cut a row (by
# the sum's length and the outputs); 8 rows stay on them
SHORT = [(H.Q4_K, 16, 2048, 6144, True), (H.Q6_K, 16, 2048, 6144, True), (H.Q4_K, 9, 2048, 4608, True),
         (H.Q5_1, 9, 2048, 3072, False), (H.Q8_0, 9, 2048, 4096, False), (H.Q6_K, 17, 2048, 2048, False),
         (H.MXFP4, 9, 768, 6000, False), (H.Q4_0, 24, 8192, 2048, True), (H.Q5_1, 13, 8192, 2048, False),
         (H.Q6_K, 33, 1280, 2048, False), (H.Q5_0, 79, 1024, 1300, True), (H.Q4_0, 8, 2048, 8192, False),
         (H.Q4_0, 9, 256, 64, True), (H.Q5_1, 16, 512, 4415, False), (H.Q5_1, 16, 512, 4416, True),
         (H.Q6_K, 64, 256, 2127, False), (H.Q6_K, 64, 256, 2128, True), (H.Q8_0, 16, 1024, 1023, False),
         (H.Q8_0, 16, 1024, 1024, True), (H.Q5_0, 40, 768, 1561, False), (H.Q5_0, 40, 768, 1562, True),
         (H.Q6_K, 43, 1280, 2000, False), (H.Q6_K, 43, 1280, 2001, True), (H.Q5_1, 64, 3072, 1007, False),
         (H.Q5_1, 64, 3072, 1008, True), (H.Q4_0, 9, 4096, 3185, False), (H.Q4_0, 9, 4096, 3186, True),
         (H.Q8_0, 32, 4096, 1695, False), (H.Q8_0, 32, 4096, 1696, True), (H.Q6_K, 9, 8192, 3299, False),
         (H.Q6_K, 9, 8192, 3300, True), (H.Q6_K, 20, 1792, 2559, False), (H.Q6_K, 20, 1792, 2560, True),
         (H.Q5_1, 16, 1376, 1855, False), (H.Q5_1, 16, 1376, 1856, True), (H.Q5_1, 9, 416, 100, True)]


@pytest.mark.parametrize("dtype,rows,cols,out,gemm", SHORT)
def test_short_batches(ctx, dtype, rows, cols, out, gemm):
    if ctx.info()[2] != 256:
        pytest.skip("the lines lie at other sizes on another number of CUs")
    x = np.random.default_rng(rows + out).standard_normal((rows, cols)).astype(np.float32)
    w = H.synth_blocks(dtype, out, cols, rows + cols, -8, -4)
    ctx.kernel_timer("ge", 16)
    got = ctx.linear(x, w, dtype, out, mode=H.MODE_Q8)
    names = list(ctx.kernel_timer_report())
    ctx.kernel_timer(None)
    assert len(names) == 1 and names[0].startswith("gemm_") == gemm, names
    same(got, O.linear(x, w, dtype, out, None))


@pytest.mark.parametrize("dtype", BLOCK[:5], ids=[H.NAMES[t] for t in BLOCK[:5]])
@pytest.mark.parametrize("rows", [16, 96])
def test_subnormal_scales(ctx, dtype, rows):
    """The products of a row's and a weight's scale are formed from halves on the
    matrix cores: scales below the least normal half (activations below
    0.0078, MXFP4 exponents up to 112) keep every bit."""
    cols, out = 1024, 9000
    rng = np.random.default_rng(dtype)
    x = rng.standard_normal((rows, cols)).astype(np.float32)
    x *= 10.0 ** -rng.uniform(1, 6.5, (rows, cols // 32)).astype(np.float32).repeat(32, 1)
    bv, bs = H.BLOCK[dtype]
    b = rng.integers(0, 256, (out, cols // bv, bs), dtype=np.uint8)
    if dtype == H.MXFP4:
        b[..., 0] = rng.integers(104, 114, b.shape[:2])
    else:
        for i in range(0, 4 if dtype == H.Q5_1 else 2, 2):
            b[..., i:i + 2] = rng.integers(1, 2048, b.shape[:2]).astype(np.uint16)[..., None].view(np.uint8)
    w = b.reshape(-1)
    ctx.kernel_timer("ge", 16)
    got = ctx.linear(x, w, dtype, out, mode=H.MODE_Q8)
    names = list(ctx.kernel_timer_report())
    ctx.kernel_timer(None)
    assert len(names) == 1 and names[0].startswith("gemm_"), names
    ref = O.linear(x, w, dtype, out)
    assert np.count_nonzero(ref) > 0.9 * ref.size
    same(got, ref)


@pytest.mark.parametrize("dtype", [H.Q4_K, H.Q8_0, H.F32], ids=["Q4_K", "Q8_0", "F32"])
def test_rows_beside_others(ctx, dtype):
    # the rows beside a row choose the tiles and the parts of its sum (here 4
    # for the 32 rows alone, 1 among 600), which changes the order of a double sum
    # and no more
    rows, cols, out = 600, 2048, 5000
    x = np.random.default_rng(7).standard_normal((rows, cols)).astype(np.float32)
    w = H.synth_normal(dtype, out, cols, 5, 0.5) if dtype == H.F32 else H.synth_blocks(dtype, out, cols, 5, -8, -4)
    whole = ctx.linear(x, w, dtype, out, mode=H.MODE_Q8)
    same(ctx.linear(x[64:96], w, dtype, out, mode=H.MODE_Q8), whole[64:96])


def test_quantized_input_and_rows_apart(ctx):
    # a row's result does not depend on who quantized it, nor on the rows beside
    # it while they leave the parts of its sum alone
    rows, cols, out = 75, 1024, 2500
    x = np.random.default_rng(3).standard_normal((rows, cols)).astype(np.float32)
    w = H.synth_blocks(H.Q4_K, out, cols, 5, -8, -4)
    dw = ctx.weight(w, H.Q4_K, out, cols)
    L = H.lib()
    dx, y, q = ctx.array(x), ctx.alloc(rows * out * 4), ctx.alloc(rows * int(L.ihip_q8_bytes(cols, 1)))
    H.check(L.ihip_enqueue_quantize(ctx.h, dx.ptr, rows, cols, 1, q.ptr, 0))
    H.check(L.ihip_enqueue_linear_at(ctx.h, q.ptr, rows, cols, H.Q4_K, dw, out, y.ptr, 0,
                                     H.MODE_Q8 | 2))
    ctx.sync()
    a = y.download(np.float32, rows * out).reshape(rows, out)
    assert np.array_equal(a, ctx.linear(x, w, H.Q4_K, out, mode=H.MODE_Q8))
    assert np.array_equal(a[32:64], ctx.linear(x[32:64], w, H.Q4_K, out, mode=H.MODE_Q8))


# float weights (gemm_flt: tiles of 32 and 64 rows, the sum split over blocks
# where there are few tiles): (rows, in, out) at the edges of tiles, chunks
# of 32 values and splits
FLOAT_SHAPES = [(4, 4096, 3100), (8, 3104, 1025), (17, 32, 33), (32, 1024, 129), (33, 1056, 65),
                (64, 2080, 40), (65, 96, 4097), (200, 2880, 31)]


@pytest.mark.parametrize("dtype", [H.F32, H.BF16, H.F16], ids=["F32", "BF16", "F16"])
def test_float_tiles_match_oracle(ctx, dtype):
    for rows, cols, out in FLOAT_SHAPES:
        rng = np.random.default_rng(rows + out)
        x = rng.standard_normal((rows, cols)).astype(np.float32)
        bias = rng.standard_normal(out).astype(np.float32)
        w = H.synth_normal(dtype, out, cols, rows + cols, 0.5)
        got = ctx.linear(x, w, dtype, out, bias, mode=H.MODE_Q8)
        ref = O.linear(x, w, dtype, out, bias)
        bits = np.abs(got.view(np.int32).astype(np.int64) - ref.view(np.int32).astype(np.int64))
        near = np.abs(got - ref) <= np.abs(ref) * 2.0 ** -23 + 1e-30
        assert np.all((bits <= 1) | near), (rows, cols, out, int(bits.max()))
        assert (bits > 0).mean() <= 1e-3
