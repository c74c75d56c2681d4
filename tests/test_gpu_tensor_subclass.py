"""Outputs of the op surface that have an operand's layout are of that operand's type, as
torch.empty_like gives it for a subclass of torch.Tensor (and plain tensors for a Parameter)."""

from __future__ import annotations

import pytest
import torch

from test_gpu_backward import pc  # noqa: F401

pytestmark = pytest.mark.gpu


class Sub(torch.Tensor):
    pass


def _ones(*shape):
    return torch.ones(*shape, device="cuda")


@pytest.mark.parametrize("kind", [Sub, torch.nn.Parameter])
def test_results_take_the_operands_type(pc, kind):  # noqa: F811
    def of(*shape):
        return _ones(*shape).as_subclass(Sub) if kind is Sub else torch.nn.Parameter(_ones(*shape))

    want = Sub if kind is Sub else torch.Tensor
    cos = sin = _ones(3, 32)
    idx = torch.zeros(2, 1, dtype=torch.int64, device="cuda")
    slots = torch.zeros(2, 1, dtype=torch.int32, device="cuda")
    slots[1] = 1
    bf = torch.ones(2, 1, device="cuda").to(torch.bfloat16)
    got = {
        "rmsnorm": pc.rmsnorm_forward(of(2, 8), of(8), 1e-6)[0],
        "conv": pc.causal_depthwise_conv1d_k4_forward(of(1, 2, 8), of(8, 4)),
        "rmsnorm dx": pc.rmsnorm_backward(_ones(2, 8), of(2, 8), of(8), _ones(2))[0],
        "rmsnorm dw": pc.rmsnorm_backward(_ones(2, 8), of(2, 8), of(8), _ones(2))[1],
        "qk dw": pc.qk_rmsnorm_rope_backward(_ones(1, 2, 3, 64), _ones(1, 2, 3, 64), of(2, 64),
                                             _ones(6), cos, sin, 3)[1],
        "gate": pc.fused_attn_gate_backward(_ones(1, 3, 128), of(1, 2, 3, 64), _ones(1, 3, 2))[0],
        "swiglu": pc.fused_swiglu_backward(_ones(2, 4), of(2, 8), 4),
        "conv dx": pc.causal_depthwise_conv1d_k4_backward(_ones(1, 2, 8), of(1, 2, 8), of(8, 4))[0],
        "conv dw": pc.causal_depthwise_conv1d_k4_backward(_ones(1, 2, 8), of(1, 2, 8), of(8, 4))[1],
        "router": pc.moe_router_topk_backward(bf, of(2, 4), idx),
        "combine": pc.moe_combine_backward(_ones(2, 8), of(1, 2, 8), idx, bf, slots)[0],
    }
    assert {k: type(v) for k, v in got.items()} == {k: want for k in got}
    assert torch.equal(got["rmsnorm"].as_subclass(torch.Tensor),
                       pc.rmsnorm_forward(_ones(2, 8), _ones(8), 1e-6)[0])
    assert torch.equal(got["combine"].as_subclass(torch.Tensor), _ones(1, 2, 8))
