"""The prompt attention over tiles of 16 rows (ops.hip attention_mfma_*): row
counts and contexts at the edges of its tiles (16 rows) and ranges (128 keys,
144 in one piece), windows that end inside a range, sinks, few tiles (the
ranges in groups and a merge) and many (no merge), heads of 64, 128 and 256,
half and float keys, values and keys that are not finite, against the CPU
oracle.

Bound: products and sums in double on both sides, e^x within an ulp of double;
only their order differs, about 1e-15 relative for sums of 2000 weights before
the one rounding to single: 2e-7 of the largest output allows two ulps."""
import numpy as np
import pytest

import infer_hip as H
import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = H.Context(0)
    yield c
    c.close()


CASES = [  # heads, kv heads, head size, rows, past, window, sinks, half
    (8, 2, 128, 2, 0, 0, False, True), (8, 2, 128, 16, 128, 0, False, True),
    (4, 1, 128, 17, 127, 0, True, True), (8, 8, 128, 33, 1000, 0, False, False),
    (8, 2, 64, 15, 129, 128, True, True), (16, 4, 64, 200, 300, 128, True, True),
    (8, 2, 64, 144, 0, 16, False, False), (2, 1, 256, 31, 0, 0, False, True),
    (4, 2, 256, 130, 513, 0, False, True), (4, 4, 256, 40, 700, 100, True, False),
    (32, 4, 128, 600, 0, 0, False, True), (64, 8, 64, 150, 50, 0, False, False),
    (8, 2, 256, 520, 0, 1024, False, True), (1, 1, 64, 3, 4000, 0, True, True)]


@pytest.mark.parametrize("heads,kvh,hd,rows,past,window,sinks,half", CASES)
def test_tiles_match_oracle(ctx, heads, kvh, hd, rows, past, window, sinks, half):
    rng = np.random.default_rng(heads * rows + past)
    total = past + rows
    q = (rng.standard_normal((rows, heads * hd)) * 2).astype(np.float32)
    k = rng.standard_normal((total, kvh * hd)).astype(np.float32)
    v = rng.standard_normal((total, kvh * hd)).astype(np.float32)
    k[total // 2] *= 8  # a key far above the others, in the middle of the ranges
    if half:
        k, v = k.astype(np.float16), v.astype(np.float16)
    sk = rng.standard_normal(heads).astype(np.float32) if sinks else None
    dq, dk, dv, y = ctx.array(q), ctx.array(k), ctx.array(v), ctx.alloc(q.nbytes)
    ds = ctx.array(sk) if sinks else None
    H.check(H.lib().ihip_enqueue_attention(ctx.h, dq.ptr, dk.ptr, dv.ptr, y.ptr, rows, heads, kvh,
                                           hd, past, window, ds.ptr if ds else 0, 0.0, int(half)))
    ctx.sync()
    got = y.download(np.float32, rows * heads * hd).reshape(rows, heads * hd)
    ref = O.causal_attention(q, heads, hd, k.astype(np.float32), v.astype(np.float32), past, kvh,
                             window, sk)
    assert np.abs(got - ref).max() <= 2e-7 * np.abs(ref).max()


# heads, kv heads, head size, rows, past, window, half, and the kernels that run:
# tiles with and without a merge, rows on their own (few rows of half-float heads
# of 256)
ROUTES = [
    (32, 4, 128, 100, 60, 0, True, "mfma"), (14, 2, 64, 200, 0, 0, False, "mfma"),
    (8, 2, 128, 100, 60, 0, True, "mfma"), (8, 2, 128, 33, 200, 0, True, "mfma merge"),
    (4, 2, 128, 20, 120, 0, False, "mfma"), (16, 8, 128, 100, 2000, 0, True, "mfma merge"),
    (16, 8, 128, 250, 60, 0, True, "mfma"), (8, 2, 256, 150, 2000, 0, True, "mfma merge"),
    (16, 8, 256, 250, 400, 0, False, "mfma merge"), (14, 2, 64, 20, 400, 128, True, "mfma"),
    (4, 2, 64, 20, 700, 300, True, "mfma merge"), (16, 8, 256, 10, 500, 0, True, "mfma merge"),
    (14, 2, 64, 300, 2000, 0, True, "mfma merge"), (8, 2, 256, 8, 500, 0, True, "part merge"),
    (8, 2, 256, 8, 500, 0, False, "mfma merge"), (8, 2, 256, 8, 2000, 1024, True, "part merge"),
    (8, 2, 256, 16, 2000, 128, True, "part merge"), (8, 2, 256, 64, 60, 0, True, "mfma"),
    (16, 8, 256, 20, 500, 0, True, "mfma merge"), (8, 2, 256, 9, 0, 0, True, "mfma")]


@pytest.mark.parametrize("heads,kvh,hd,rows,past,window,half,names", ROUTES)
def test_routes_match_oracle(ctx, heads, kvh, hd, rows, past, window, half, names):
    if ctx.info()[2] != 256:
        pytest.skip("the lines lie at other sizes on another number of CUs")
    ctx.kernel_timer("attention_", 16)
    test_tiles_match_oracle(ctx, heads, kvh, hd, rows, past, window, False, half)
    got = [k.split("_")[1] for k in ctx.kernel_timer_report()]
    ctx.kernel_timer(None)
    assert " ".join(got) == names


# heads, kv heads, head size, rows, past, window, sinks, half, and where: the
# key rows that hold infinities or a NaN (of the total), in the values or keys
ODD = [
    (4, 2, 256, 20, 0, 0, False, True, "v", (5, 19)), (4, 2, 256, 33, 300, 0, False, False, "v", (301, 332)),
    (2, 1, 128, 40, 100, 64, True, True, "v", (90, 120)), (8, 2, 128, 17, 0, 0, False, False, "v", (16,)),
    (4, 4, 64, 48, 0, 0, False, True, "v", (20, 40)), (4, 1, 64, 31, 500, 128, True, False, "v", (380, 515)),
    (8, 8, 256, 300, 0, 0, False, True, "v", (130, 299)), (40, 8, 128, 250, 0, 0, False, True, "v", (7, 140)),
    (4, 2, 256, 20, 200, 0, False, True, "k", (10, 210)), (2, 2, 256, 18, 900, 0, True, False, "k", (901,)),
    (4, 2, 128, 25, 300, 0, False, False, "k", (0, 310)), (8, 4, 64, 20, 150, 32, False, True, "k", (140, 165)),
    (40, 8, 128, 250, 0, 0, False, True, "k", (128, 200))]


@pytest.mark.parametrize("heads,kvh,hd,rows,past,window,sinks,half,where,at", ODD)
def test_infinities_and_nan_reach_the_rows_that_see_them(ctx, heads, kvh, hd, rows, past, window, sinks,
                                                         half, where, at):
    """A value or key that is not finite changes the rows that see its key as it
    changes them on the CPU, and no other row, whatever rows share its tile."""
    rng = np.random.default_rng(rows + past + hd)
    total = past + rows
    q = rng.standard_normal((rows, heads * hd)).astype(np.float32)
    k = rng.standard_normal((total, kvh * hd)).astype(np.float32)
    v = rng.standard_normal((total, kvh * hd)).astype(np.float32)
    odd = v if where == "v" else k
    for i, r in enumerate(at):
        odd[r, (3 + 5 * i) % hd::hd] = (np.inf, np.nan)[i % 2] if where == "v" else (-np.inf, np.nan)[i % 2]
        odd[r, (hd // 2 + i)] = np.inf
    if half:
        k, v = k.astype(np.float16), v.astype(np.float16)
    sk = rng.standard_normal(heads).astype(np.float32) if sinks else None
    dq, dk, dv, y = ctx.array(q), ctx.array(k), ctx.array(v), ctx.alloc(q.nbytes)
    ds = ctx.array(sk) if sinks else None
    H.check(H.lib().ihip_enqueue_attention(ctx.h, dq.ptr, dk.ptr, dv.ptr, y.ptr, rows, heads, kvh,
                                           hd, past, window, ds.ptr if ds else 0, 0.0, int(half)))
    ctx.sync()
    got = y.download(np.float32, rows * heads * hd).reshape(rows, heads * hd)
    with np.errstate(all="ignore"):
        ref = O.causal_attention(q, heads, hd, k.astype(np.float32), v.astype(np.float32), past, kvh,
                                 window, sk)
    assert not np.isfinite(ref).all() and np.isfinite(ref).any()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    ok = np.isfinite(ref)
    assert np.abs(got[ok] - ref[ok]).max() <= 2e-7 * np.abs(ref[ok]).max()
