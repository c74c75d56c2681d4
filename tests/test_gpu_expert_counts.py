"""Rows per expert of the last step: the counters' spread copy, as read back, against the
router's choices of the same step (exact), on every kernel the router and the expert GEMMs
switch to with the number of rows."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from pulsar_engine import weights as W
from pulsar_engine.config import small_config
from pulsar_engine.engine import HipEngine
from pulsar_engine.model import DeviceModel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("batch", [1, 9, 40, 70])
def test_counts_are_the_routers(dtype, batch):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    cfg = small_config(n_heads=16, n_kv_heads=4)
    model = DeviceModel(cfg, W.synthetic_state(cfg, seed=3), dtype)
    ids = np.stack([W.uniform_ids(b, "counts", 20, cfg.vocab_size) for b in range(batch)])
    with HipEngine(model, batch=batch, max_prompt=20, max_new=12, temperature=0.0,
                   stop_ids=[]) as eng:
        eng.prefill(ids)
        eng.step(4)
        idx, got = eng.topk_idx(), eng.expert_counts()
    assert idx.shape[1] > 0
    for layer in range(cfg.n_core):
        want = np.bincount(idx[layer].ravel(), minlength=cfg.n_routed_experts)
        np.testing.assert_array_equal(got[layer], want)
