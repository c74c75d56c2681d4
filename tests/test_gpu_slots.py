"""GPU parity of moe_slots_from_order: the one-workgroup launch of short assignment lists and
the counted launches of long ones, on both sides of the line between them."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pc():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import pulsar_cuda

    return pulsar_cuda


@pytest.mark.parametrize("E", [1, 16, 1024])
@pytest.mark.parametrize("M", [1, 1024, 8192, 8193, 70001])
def test_slots_counts(pc, M, E):
    """Counts and ranks of both slot paths against a stable sort, with dropped ids outside
    [0, E) in the flat list (their slot is -1; they sort to the ends of the order)."""
    g = torch.Generator().manual_seed(M + E)
    flat = torch.randint(0, E, (M,), generator=g)
    if M > 100:
        flat[::97] = E  # past the last expert: sorts last
    order = torch.argsort(flat, stable=True)
    C = max(1, M // (2 * E))
    slots, counts = pc.moe_slots_from_order(flat.cuda(), order.cuda(), E, C)
    want = torch.bincount(flat, minlength=E + 1)
    start = want.cumsum(0) - want
    rank = torch.empty(M, dtype=torch.int64)
    rank[order] = torch.arange(M) - start[flat[order]]
    rank[(rank >= C) | (flat >= E)] = -1
    assert torch.equal(slots.cpu().long(), rank)
    assert torch.equal(counts.cpu(), want[:E])
