"""The mid-size projection GEMMs against the row-tile ones, bit for bit (both add the same 8
chunks of K in the same order), at widths and row counts around their lines: K of 256 (every
k tile a chunk of its own; with a shared expert twice as wide the two k tiles of a stage lie
apart), 512 and 1024, shared experts of the routed width and twice that, one row more and
less than whole 64-row tiles, and a number of heads whose gate columns end a column block
short."""

from __future__ import annotations

import os

import numpy as np
import pytest
import torch

from pulsar_engine import weights as W
from pulsar_engine.config import small_config
from pulsar_engine.engine import HipEngine
from pulsar_engine.model import DeviceModel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,batch", [
    (dict(d_model=256, d_expert=256, d_shared=256), 65),
    (dict(d_model=256, d_expert=256, d_shared=512), 63),
    (dict(d_model=512, d_expert=256, d_shared=512), 1),
    (dict(d_model=1024, d_expert=512, d_shared=1024), 129),
    (dict(d_model=512, d_expert=1024, d_shared=1024), 64),
])
def test_mid_equals_row_tiles(dims, batch):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    cfg = small_config(n_heads=16, n_kv_heads=4, **dims)
    model = DeviceModel(cfg, W.synthetic_state(cfg, seed=11), torch.bfloat16)
    ids = np.stack([W.uniform_ids(b, "mid_widths", 9, cfg.vocab_size) for b in range(batch)])
    out = {}
    old = os.environ.get("PULSAR_GEMM_MID_ROWS")
    try:
        for mid in (0, 1):
            os.environ["PULSAR_GEMM_MID_ROWS"] = str(mid)
            print(f"[mid widths] {dims} batch={batch} mid_rows={mid}", flush=True)
            with HipEngine(model, batch=batch, max_prompt=9, max_new=6, temperature=0.0,
                           stop_ids=[]) as eng:
                eng.prefill(ids)
                eng.step(5)
                out[mid] = eng.tokens(), eng.logits(batch).copy()
    finally:
        if old is None:
            os.environ.pop("PULSAR_GEMM_MID_ROWS", None)
        else:
            os.environ["PULSAR_GEMM_MID_ROWS"] = old
    assert np.isfinite(out[0][1]).all()
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1], out[1][1])
