"""The rotary rows formed on the device (ops.hip rotary_rows): prompt chunks and
the decode steps after them against the CPU oracle, whose angles, cosines and
sines are the host's, for the whole head, a partial rotation (Qwen3.5), YaRN's
scale (gpt-oss) and two sets (Gemma 4), with positions across a chunk.

Bound: a cosine or sine in double rounds to the same single on both sides but
where the two math libraries' last double bits straddle a rounding (1e-9 of
the values), so the logits agree to single rounding (1e-5, the bound of the
other device tests)."""
import numpy as np
import pytest

import infer_hip as H
import oracle_lib as O
from infer_hip import models

pytestmark = pytest.mark.gpu

SMALL = dict(layers=2, vocab=512, hidden=256)
CFGS = {
    "whole": models.tiny("qwen3-0.6b-q8_0", heads=2, kv_heads=1, head_dim=128, ffn=256, **SMALL),
    "small-theta": models.tiny("qwen3-0.6b-q8_0", heads=4, kv_heads=2, head_dim=64, ffn=256,
                               rope_theta=30.0, **SMALL),
    "yarn": models.tiny("gpt-oss-20b-mxfp4", heads=4, kv_heads=2, head_dim=64, experts=4,
                        experts_used=2, expert_ffn=256, **SMALL),
    "partial": models.tiny("qwen35-0.8b-q8_0", heads=2, kv_heads=1, head_dim=64, rope_dims=22,
                           interval=1, ffn=256, lin_key_heads=1, lin_value_heads=1, **SMALL),
    "two-sets": models.tiny("gemma4-26b-a4b-q8_0", heads=2, kv_heads=2, head_dim=64,
                            full_head_dim=128, full_kv_heads=1, rope2_pairs=16, pattern=2,
                            ffn=256, experts=4, experts_used=2, expert_ffn=256, **SMALL),
}


@pytest.fixture(scope="module")
def ctx():
    c = H.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("name", list(CFGS))
def test_positions_match_oracle(ctx, name):
    s = models.Spec(CFGS[name], seed=9, sigma=0.05)
    ids = (np.arange(141, dtype=np.int32) * 53 + 7) % 512
    dev, cpu = H.Model(ctx, s, max_tokens=32), O.Model(s, 256)
    for part in (ids[:1], ids[1:134], ids[134:]):
        a, b = dev.forward(part, all_logits=True), cpu.forward(part, all_logits=True)
        assert float(np.abs(a - b).max() / np.abs(b).max()) < 1e-5
    # the decode's table of positions: the ids drawn from here on
    first = int(np.argmax(b[-1]))
    got = dev.decode(first, 9)
    want, at = [], first
    for _ in range(9):
        at = int(np.argmax(cpu.forward([at])))
        want.append(at)
    assert got.tolist() == want
    dev.close()
    cpu.close()
