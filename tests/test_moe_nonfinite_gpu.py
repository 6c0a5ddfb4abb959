"""Router logits that are not finite: a row with a NaN or +inf, or with nothing but -inf, has no softmax.  Its
token still gets top_k different experts, with NaN weights, and every other token keeps its result."""

import pytest
import torch

from anna_amd import fused_ops
from anna_amd.moe import SparseMoeInt4
from tests.test_moe_gpu import make_bank

pytestmark = pytest.mark.gpu


def spoil(logits):
    """(logits with three rows that have no softmax and one with a -inf that has, mask of the three)"""
    bad = logits.clone()
    bad[1, 2] = float("nan")
    bad[3, -1] = float("inf")
    bad[4] = float("-inf")
    bad[6, 0] = float("-inf")
    mask = torch.zeros(logits.shape[0], dtype=torch.bool, device=logits.device)
    mask[[1, 3, 4]] = True
    return bad, mask


# experts per lane: one, two, four and sixteen; a count that is no multiple of 4
@pytest.mark.parametrize("experts,top_k", [(7, 3), (16, 16), (128, 8), (254, 5), (512, 64)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_router_rows_without_a_softmax(gpu, experts, top_k, dtype):
    torch.manual_seed(experts)
    clean = torch.randn(9, experts, device=gpu).to(dtype)
    bad, mask = spoil(clean)
    clean[6, 0] = float("-inf")
    w, sel, usage = fused_ops.moe_router(bad, top_k)
    cw, csel, _ = fused_ops.moe_router(clean, top_k)
    assert all(len(set(r)) == top_k and 0 <= min(r) and max(r) < experts for r in sel.tolist())
    assert torch.equal(usage.long(), torch.bincount(sel.flatten(), minlength=experts))
    assert torch.equal(w[~mask], cw[~mask]) and torch.equal(sel[~mask], csel[~mask])
    assert bool(torch.isnan(w[mask]).all())


# the routing in one launch, the separate router and dispatch, and the form for many routes per expert
@pytest.mark.parametrize("tokens,experts,top_k", [(9, 16, 4), (60, 64, 4), (75, 16, 4), (150, 16, 4)])
def test_block_keeps_the_other_tokens(gpu, tokens, experts, top_k):
    torch.manual_seed(tokens)
    bank = make_bank(experts, 256, 256, 128, torch.float32, gpu, tokens)
    x = torch.randn(tokens, 256, device=gpu, dtype=torch.bfloat16)
    clean = torch.randn(tokens, experts, device=gpu)
    bad, mask = spoil(clean)
    clean[6, 0] = float("-inf")
    block = SparseMoeInt4(bank, num_experts=experts, top_k=top_k)
    got, want = block(x, bad), block(x, clean)
    assert bool(torch.isnan(got[mask]).all())
    assert torch.equal(got[~mask], want[~mask])
