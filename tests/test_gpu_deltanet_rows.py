"""The Gated DeltaNet of prompt chunks (deltanet.hip dn_convprep, dn_rule_128,
dn_rule_256) against the CPU oracle: key and value sizes at and around the
kernels' tiles (a column's 32 lanes and pairs, 8 columns a block, 16 or 8
tokens a chunk), convolutions of 1 to 5 (and 8: the general kernels), row
counts at the chunk edges, the state carried into a second chunk.

Bound: both sides round to single at the same steps and hold every sum in
double, so a value differs only where a double sum's order moves a single
rounding; such a value moves an activation code of a later product by one of
127 steps at most, 1e-2 of that product's largest term; without a moved code
the logits agree to single rounding. 1e-5 asks for the second on these inputs
(the reference's own device bound)."""
import numpy as np
import pytest

import infer_hip as H
import oracle_lib as O
from infer_hip import models

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = H.Context(0)
    yield c
    c.close()


def spec(dk, dv, kh, vh, kw):
    cfg = models.tiny("qwen35-0.8b-q8_0", layers=2, vocab=512, hidden=256, ffn=256, heads=4,
                      kv_heads=2, head_dim=64, rope_dims=16, interval=3, lin_key_heads=kh,
                      lin_value_heads=vh, lin_key_dim=dk, lin_value_dim=dv, lin_conv=kw)
    return models.Spec(cfg, seed=dk + dv + kw, sigma=0.05)


@pytest.mark.parametrize("dk,dv,kh,vh,kw,rows,more", [
    (128, 128, 2, 2, 4, 16, 17), (128, 128, 1, 2, 4, 8, 1), (64, 32, 2, 2, 2, 9, 2),
    (96, 64, 1, 1, 5, 33, 3), (256, 256, 1, 1, 3, 8, 9), (200, 96, 1, 2, 4, 25, 5),
    (130, 32, 1, 1, 1, 17, 8), (2, 32, 2, 2, 4, 3, 7), (128, 160, 1, 1, 8, 12, 4),
    (32, 288, 1, 1, 4, 10, 9)])
def test_rows_match_oracle(ctx, dk, dv, kh, vh, kw, rows, more):
    s = spec(dk, dv, kh, vh, kw)
    ids = (np.arange(rows + more, dtype=np.int32) * 37 + 11) % 512
    dev, cpu = H.Model(ctx, s, max_tokens=128), O.Model(s, 128)
    for part in (ids[:rows], ids[rows:]):
        a, b = dev.forward(part, all_logits=True), cpu.forward(part, all_logits=True)
        assert float(np.abs(a - b).max() / np.abs(b).max()) < 1e-5
    dev.close()
    cpu.close()
