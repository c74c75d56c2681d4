"""The prefill kernels' tile shapes: every GEMM shape sums an output's K in the same order, and
a query's attention and a row's routing do not depend on the tile or workgroup that holds
them, so a sequence's prefill logits are the same bits in batches small and large enough to
take each shape."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from pulsar_engine import weights as W
from pulsar_engine.config import small_config
from pulsar_engine.engine import HipEngine
from pulsar_engine.model import DeviceModel

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    cfg = small_config(n_heads=16, n_kv_heads=4)
    return DeviceModel(cfg, W.synthetic_state(cfg, seed=3), torch.bfloat16)


@pytest.mark.parametrize("T", [128, 131, 193, 260])
def test_prefill_logits_do_not_depend_on_the_tile_shape(model, T):
    V = model.cfg.vocab_size
    prompts = np.stack([W.uniform_ids(b, "wide", T, V) for b in range(128)])

    def logits(B):
        with HipEngine(model, batch=B, max_prompt=T, max_new=2, temperature=0.0,
                       stop_ids=[]) as eng:
            eng.prefill(prompts[:B])
            return eng.logits(B)

    # tiles of the widest projection (1552 columns): 128 rows take 64 x 64 tiles, 2000 rows
    # 64 x 128, 4000 rows 128 x 128, 16384 rows and more 128 x 256; attention in 16, 32 and 64
    # queries; the router in 1, 4 and (260 tokens) 8 row tiles; q/k norm and RoPE row by row and,
    # from 1024 rows, 8 rows at a time (across sequences and the window's start)
    sets = {B: logits(B) for B in (1, 16, 32, 128)}
    for B, got in sets.items():
        assert np.isfinite(got).all()
        assert np.array_equal(got[:1], sets[128][:1]), B
        assert np.array_equal(got, sets[128][:B]), B
