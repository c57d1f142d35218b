"""The grouping of a prompt chunk's experts (ops.hip moe_plan: 1024 threads, each
with its experts, a scan over lanes and waves) through a layer of few experts,
of as many as lanes or threads and of more, with experts that get no slot and
experts that get more than one work item, against the CPU oracle. The order
of an expert's slots changes no row, so the bound is the model tests' (the
same roundings on both sides)."""
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


@pytest.mark.parametrize("experts,used,rows", [(3, 2, 150), (64, 4, 97), (65, 8, 200),
                                               (1024, 4, 90), (1100, 3, 96)])
def test_grouped_experts_match_oracle(ctx, experts, used, rows):
    cfg = models.tiny("gpt-oss-20b-mxfp4", layers=1, vocab=512, hidden=64, heads=2, kv_heads=1,
                      head_dim=64, experts=experts, experts_used=used, expert_ffn=64)
    s = models.Spec(cfg, seed=experts, sigma=0.1)
    ids = (np.arange(rows, dtype=np.int32) * 29 + 3) % 512
    dev, cpu = H.Model(ctx, s, max_tokens=256), O.Model(s, 256)
    a, b = dev.forward(ids, all_logits=True), cpu.forward(ids, all_logits=True)
    assert float(np.abs(a - b).max() / np.abs(b).max()) < 1e-5
    dev.close()
    cpu.close()
