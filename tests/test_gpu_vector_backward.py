"""GPU parity of the 16-byte forms of the backward ops at the edges of their chunks, tasks
and workgroups, with the bounds of test_gpu_backward (one rounding of an fp32 result for bf16
outputs, 1e-5 of the largest value for fp32 ones), and of their element forms, which take
tensors whose pointers are not 16-byte aligned."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import backward_ref as BW
from test_gpu_backward import DTYPES, _check, _np, _rand, _routing, _tables, pc  # noqa: F401

pytestmark = pytest.mark.gpu


def _off(t):
    """The same values at a pointer one element past a 16-byte boundary."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    buf[1:].copy_(t.reshape(-1))
    return buf[1:].view(t.shape)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,dim", [(1, 8), (9, 520), (8, 1024), (2049, 264), (4100, 64),
                                      (7, 2048), (3, 2056)])
def test_rmsnorm_backward_chunks(pc, rows, dim, dtype):  # noqa: F811
    x = _rand(rows, dim, seed=dim, dtype=dtype)
    w = torch.rand(dim, device="cuda") + 0.5
    _, rs = pc.rmsnorm_forward(x, w, 1e-6)
    dy = _rand(rows, dim, seed=dim + 1, dtype=dtype)
    ox, ow = BW.rmsnorm_bwd(_np(dy), _np(x), _np(w), _np(rs))
    for xx in (x, _off(x)):
        dx, dw = pc.rmsnorm_backward(dy, xx, w, rs)
        _check(dx, ox, dtype, "rmsnorm dx")
        _check(dw, ow, torch.float32, "rmsnorm dw")


def test_rmsnorm_backward_infinite_weight(pc):  # noqa: F811
    """Lanes past a row's last chunk add nothing, an infinite weight in that chunk included."""
    x = torch.rand(5, 520, device="cuda") + 0.5
    w, dy = torch.ones(520, device="cuda"), torch.ones(5, 520, device="cuda")
    w[-1] = float("inf")
    dx, dw = pc.rmsnorm_backward(dy, x, w, torch.ones(5, device="cuda"))
    assert bool((dx[:, :-1] == -float("inf")).all()), "dx = r w dy - x inf"
    assert bool(torch.isfinite(dw).all())


def test_backward_of_longer_weights(pc):  # noqa: F811
    """Gradients of weight entries that no column uses are zero."""
    x, dy = _rand(1, 6, 64, seed=1), _rand(1, 6, 64, seed=2)
    for _ in range(8):  # freed blocks hold other values
        torch.full((4096,), 7.0, device="cuda")
    w = torch.rand(96, device="cuda")
    assert not pc.rmsnorm_backward(dy, x, w, torch.ones(6, device="cuda"))[1][64:].any()
    w = torch.rand(96, 4, device="cuda")
    assert not pc.causal_depthwise_conv1d_k4_backward(dy, x, w)[1][64:].any()
    w, (cos, sin) = torch.rand(2, 1024, device="cuda"), _tables(3)
    q, dq = x.view(1, 2, 3, 64), dy.view(1, 2, 3, 64)
    sevens = [torch.full_like(w, 7.0) for _ in range(8)]
    del sevens
    dw = pc.qk_rmsnorm_rope_backward(dq, q, w, torch.ones(6, device="cuda"), cos, sin, 3)[1]
    assert dw.shape == w.shape and not dw.view(-1)[2 * 64:].any()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("B,H,T", [(1, 1, 1), (3, 4, 11), (1, 16, 65), (2, 3, 2100), (70, 16, 1)])
def test_qk_backward_groups(pc, B, H, T, dtype):  # noqa: F811
    qkv = _rand(B, T, (H + 2) * 64, seed=T, dtype=dtype)
    x = qkv[..., : H * 64].view(B, T, H, 64).transpose(1, 2)
    w = torch.rand(H, 64, device="cuda") + 0.5
    cos, sin = _tables(T)
    y, rs = pc.qk_rmsnorm_rope_forward(x, w, cos, sin, T)
    dy = _rand(*y.shape, seed=12, dtype=dtype)
    ox, ow = BW.qk_rmsnorm_rope_bwd(_np(dy), _np(x), _np(w), _np(rs), _np(cos), _np(sin))
    for d in (dy, _off(dy)):
        dx, dw = pc.qk_rmsnorm_rope_backward(d, x, w, rs, cos, sin, T)
        _check(dx, ox, dtype, "qk dx")
        _check(dw, ow, torch.float32, "qk dw")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("B,H,T", [(1, 1, 1), (3, 5, 7), (2, 16, 33)])
def test_gate_and_swiglu_backward_chunks(pc, B, H, T, dtype):  # noqa: F811
    a = _rand(B, H, T, 64, seed=21, dtype=dtype)
    gl = _rand(B, T, H, seed=22, dtype=torch.float32, scale=2.0)
    go = _rand(B, T, H * 64, seed=23, dtype=dtype)
    oa, ol = BW.attn_gate_bwd(_np(go), _np(a), _np(gl))
    gu = _rand(B * T, 2 * 8 * H, seed=H, dtype=dtype, scale=3.0)
    d = _rand(B * T, 8 * H, seed=H + 1, dtype=dtype)
    og = BW.swiglu_bwd(_np(d), _np(gu), 8 * H)
    for f in (lambda t: t, _off):
        da, dl = pc.fused_attn_gate_backward(f(go), a, gl)
        _check(da, oa, dtype, "gate d_attn")
        _check(dl, ol, torch.float32, "gate d_logits")
        _check(pc.fused_swiglu_backward(f(d), gu, 8 * H), og, dtype, "swiglu dgu")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("B,T,D", [(1, 3, 8), (5, 4, 264), (3, 5, 256), (2, 33, 1024),
                                   (40, 1, 64), (1, 1000, 1024), (2, 4099, 1032)])
def test_conv_backward_runs(pc, B, T, D, dtype):  # noqa: F811
    x = _rand(B, T, D, seed=T, dtype=dtype)
    w = _rand(D, 4, seed=T + 1, dtype=torch.float32, scale=0.5)
    dout = _rand(B, T, D, seed=T + 2, dtype=dtype)
    ox, ow = BW.conv_k4_bwd(_np(dout), _np(x), _np(w))
    for xx in (x, _off(x)):
        dx, dw = pc.causal_depthwise_conv1d_k4_backward(dout, xx, w)
        _check(dx, ox, dtype, "conv dx")
        _check(dw, ow, torch.float32, "conv dw")


@pytest.mark.parametrize("T", [2, 9])
def test_conv_backward_leaves_out_terms_past_the_ends(pc, T):  # noqa: F811
    """An infinite gradient or weight meets no zero standing for a row outside the sequence
    (the product would be NaN): dx[t] and dw[:, k] hold only the terms that exist."""
    D = 8
    x, dout = torch.ones(1, T, D, device="cuda"), torch.ones(1, T, D, device="cuda")
    w = torch.ones(D, 4, device="cuda")
    w[:, 3] = float("inf")
    dout[0, 0, 0] = float("inf")
    dx, dw = pc.causal_depthwise_conv1d_k4_backward(dout, x, w)
    assert not torch.isnan(dx).any() and not torch.isnan(dw).any()
    assert torch.isfinite(dx[0, max(0, T - 3):, 1:]).all()
    assert torch.isinf(dw[0, 0]) and torch.isfinite(dw[0, 1:]).all()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("N,D,K", [(1, 8, 1), (5, 520, 3), (33, 1024, 4), (6, 2048, 8),
                                   (7, 2056, 5), (9, 8, 4), (5, 24, 8), (6, 1032, 4)])
def test_moe_backward_chunks(pc, N, D, K, dtype):  # noqa: F811
    """Rows of whole waves and of less, down to fewer chunks than assignments (D = 8, 24)."""
    E, C = 16, max(2, int(np.ceil(N * K / 16 * 0.9)))
    idx, slots = _routing(N, K, E, C, N)
    ti, ts = torch.as_tensor(idx, device="cuda"), torch.as_tensor(slots, device="cuda")
    dei, eo = _rand(E, C, D, seed=31, dtype=dtype), _rand(E, C, D, seed=32, dtype=dtype)
    w = torch.rand(N, K, device="cuda").to(torch.bfloat16)
    dout = _rand(N, D, seed=33, dtype=dtype)
    od = BW.dispatch_bwd(_np(dei), idx, slots, N, D)
    oe, ow = BW.combine_bwd(_np(dout), _np(eo), idx, _np(w), slots)
    for f in (lambda t: t, _off):
        _check(pc.moe_dispatch_backward(f(dei), ti, ts, N, D), od, dtype, "dispatch dx")
        deo, dw = pc.moe_combine_backward(f(dout), eo, ti, w, ts)
        _check(deo, oe, dtype, "combine d_eo")
        _check(dw, ow, torch.bfloat16, "combine d_w")


def test_dropped_assignments_read_no_infinity(pc):  # noqa: F811
    """A dropped assignment contributes nothing even where row 0 of the experts' tensor, which
    its lanes read, is infinite."""
    N, D, K, E, C = 3, 64, 2, 4, 2
    ti = torch.tensor([[1, 2], [3, 1], [2, 3]], device="cuda")
    ts = torch.tensor([[-1, 0], [0, 0], [1, -1]], dtype=torch.int32, device="cuda")
    eo = torch.ones(E, C, D, device="cuda")
    eo[0] = float("inf")
    assert torch.equal(pc.moe_dispatch_backward(eo, ti, ts, N, D)[:, 0].cpu(),
                       torch.tensor([1.0, 2.0, 1.0]))
    deo, dw = pc.moe_combine_backward(torch.ones(N, D, device="cuda"), eo, ti,
                                      torch.ones(N, K, device="cuda").to(torch.bfloat16), ts)
    assert torch.equal(dw.float().cpu(), torch.tensor([[0.0, 64.0], [64.0, 64.0], [64.0, 0.0]]))
    assert torch.isfinite(deo).all()
