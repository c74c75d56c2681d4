"""fp32 prefill against the oracle around the lines between its kernels: the tiled GEMMs from
16 tokens on (32-row tiles: one row more and less than whole tiles), the row-wise attention up
to 256 tokens, prompts past the sliding window, and several sequences at once; then decoding
over more than one 256-key split. Bound: 2e-5 of the largest logit (fp32 sums of up to 768
terms through 12 layer passes, in another order than the oracle's)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import max_abs_rel
from oracle import pulsar_ref as R
from pulsar_engine import weights as W
from pulsar_engine.config import small_config
from pulsar_engine.engine import HipEngine
from pulsar_engine.model import DeviceModel

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[dict(), dict(d_expert=512, d_shared=768)])
def pair(request):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    cfg = small_config(max_seq_len=1024, **request.param)
    st = W.synthetic_state(cfg, seed=5)
    return (cfg, R.load_ref(cfg, st, torch.float32, stop_ids=set()),
            DeviceModel(cfg, st, torch.float32, rope_len=1024))


@pytest.mark.parametrize("T", [1, 15, 16, 17, 33, 64, 95, 255, 256, 257])
def test_prefill_logits(pair, T):
    cfg, ref, model = pair
    B = 2
    ids = np.stack([W.uniform_ids(b, "f32", T, cfg.vocab_size) for b in range(B)])
    with HipEngine(model, batch=B, max_prompt=T, max_new=2, temperature=0.0, stop_ids=[]) as eng:
        eng.prefill(ids)
        got = eng.logits(B)
    for b in range(B):
        want = ref.prefill(torch.as_tensor(ids[b:b + 1]), R.RefKVCache(cfg))
        err = max_abs_rel(got[b], want.reshape(-1))
        assert err < 2e-5, (T, b, err)


def test_decode_over_several_splits(pair):
    cfg, ref, model = pair
    ids = W.uniform_ids(9, "f32", 600, cfg.vocab_size)
    want = list(ref.self_speculative_ids(ids, 6, 0.0, 1.0, 10.0))
    with HipEngine(model, batch=1, max_prompt=600, max_new=6, temperature=0.0,
                   repetition_penalty=10.0, stop_ids=[]) as eng:
        eng.prefill(ids[None])
        eng.run()
        assert eng.tokens()[0] == want
