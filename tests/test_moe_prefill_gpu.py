"""The sparse block for many routes per expert (anna_mi_moe_prefill) against the fp64 brute force over the
dequantized bank, and against the separate ops' routing."""

import pytest
import torch

from anna_amd import _lib
from anna_amd.moe import SparseMoeInt4
from tests._util import BF16_TOL, rel_err
from tests.test_moe_gpu import dequant_experts, make_bank

pytestmark = pytest.mark.gpu


def brute_force(bank, x, logits, top_k, norm):
    # (as cp.moe_route, with equal logits in the order of their experts: 16-bit ones have some)
    w, sel = (t[:, :top_k] for t in torch.softmax(logits.cpu(), dim=-1, dtype=torch.float32).sort(
        dim=-1, descending=True, stable=True))
    w = w / w.sum(dim=-1, keepdim=True) if norm else w
    out = torch.zeros(x.shape, dtype=torch.float64)
    experts = dequant_experts(bank, sorted(set(sel.reshape(-1).tolist())))
    xd = x.cpu().double()
    for e, (wg, wu, wd) in experts.items():
        t, k = (sel == e).nonzero(as_tuple=True)
        g, u = xd[t] @ wg.double().t(), xd[t] @ wu.double().t()
        out.index_add_(0, t, (torch.nn.functional.silu(g) * u) @ wd.double().t() * w[t, k].double().unsqueeze(1))
    return out.numpy()


# fp16 states: the activation between the products is rounded to bf16 (2^-9 of each element at most, so
# 1.1e-3 of a sum of many in 2-norm; 1.7e-3 measured with the other roundings); the largest error over the
# largest value is allowed about twice that
FP16_TOL = 4e-3


def takes_prefill(bank, x, logits, top_k):
    """Whether the dispatch rule sends the call to the form tested here."""
    a = _lib.MoePrefillArgs()
    a.dtype, a.logits_dtype, a.scale_dtype = (_lib.dtype_code(t.dtype) for t in (x, logits, bank.gate_qscale))
    a.tokens, a.num_experts, a.top_k, a.group_size = x.shape[0], logits.shape[1], top_k, bank.group_size
    a.hidden_dim, a.intermediate_dim = bank.hidden_dim, bank.intermediate_dim
    a.hidden, a.hidden_row_stride = x.data_ptr(), x.stride(0)
    a.gate_qweight, a.up_qweight, a.down_qweight = (t.data_ptr() for t in (bank.gate_qweight, bank.up_qweight,
                                                                         bank.down_qweight))
    a.hidden_packed_cols, a.hidden_groups = bank.gate_qweight.shape[2], bank.gate_qscale.shape[1]
    a.intermediate_packed_cols, a.intermediate_groups = bank.down_qweight.shape[2], bank.down_qscale.shape[1]
    return _lib.load().anna_mi_moe_prefill_workspace(a) > 0


@pytest.fixture
def forced(monkeypatch):
    """The form on every shape it can compute, faster there or not."""
    monkeypatch.setenv("ANNA_MI_MOE_FORM", "P")


# sweeps of one to three chunks, several sweeps, a ragged last tile
# (intermediate 384 = 3 x 128, hidden 384 = 1.5 x 256), one group of K, the most groups of K, one
# token per wave and several, tokens past one workgroup's share
@pytest.mark.parametrize("tokens,experts,top_k,hidden,inter,dtype,scales,norm", [
    (73, 4, 1, 128, 128, torch.bfloat16, torch.float32, True),
    (75, 8, 2, 256, 384, torch.float16, torch.float32, True),
    (200, 16, 4, 384, 256, torch.bfloat16, torch.bfloat16, False),
    (333, 32, 8, 1024, 128, torch.bfloat16, torch.float16, True),
    (130, 8, 8, 512, 640, torch.float16, torch.bfloat16, True),
    (100, 8, 2, 4096, 128, torch.bfloat16, torch.float32, True),
    (5003, 3, 1, 128, 128, torch.bfloat16, torch.float32, True),
    (40, 64, 64, 256, 128, torch.bfloat16, torch.float32, False),
])
def test_prefill_block_matches_brute_force(gpu, forced, tokens, experts, top_k, hidden, inter, dtype, scales, norm):
    bank = make_bank(experts, hidden, inter, 128, scales, gpu, tokens)
    torch.manual_seed(tokens)
    wide = torch.randn(tokens, hidden + 64, device=gpu).to(dtype)
    x = wide[:, :hidden]  # rows a stride apart
    logits = torch.randn(tokens, experts, device=gpu)
    block = SparseMoeInt4(bank, num_experts=experts, top_k=top_k, norm_topk_prob=norm)
    tol = BF16_TOL if dtype == torch.bfloat16 else FP16_TOL
    for lg in (logits, logits.to(dtype)):  # (16 bits: the reference's own logits)
        assert takes_prefill(bank, x, lg, top_k)
        ref = brute_force(bank, x, lg, top_k, norm)
        assert rel_err(block(x, lg).double().cpu().numpy(), ref) <= tol


def test_prefill_block_skewed_experts(gpu):
    """Experts without routes, one with a single route and one with nearly all of them (more sweeps than
    workgroups were launched for)."""
    experts, hidden, inter, tokens = 16, 256, 256, 700
    bank = make_bank(experts, hidden, inter, 128, torch.float32, gpu, 1)
    torch.manual_seed(5)
    x = torch.randn(tokens, hidden, device=gpu, dtype=torch.bfloat16)
    logits = torch.full((tokens, experts), -30.0, device=gpu)
    logits[:, 3] = 5.0
    logits[:, 9] = 4.0 + torch.rand(tokens, device=gpu) * 0.5
    logits[17, 12] = 9.0
    block = SparseMoeInt4(bank, num_experts=experts, top_k=2)
    assert takes_prefill(bank, x, logits, 2)
    got = block(x, logits)
    assert rel_err(got.double().cpu().numpy(), brute_force(bank, x, logits, 2, True)) <= BF16_TOL
    assert torch.equal(got, block(x, logits))  # no atomics: the same bits again


def test_prefill_takes_only_its_shapes(gpu):
    """Group 64, fp32 hidden states and rows that are not 16-byte aligned go the general way, and so do shapes
    on which it is the faster one: both sides of each line of the rule."""
    torch.manual_seed(2)
    for experts, hidden, inter, group, dtype, tokens, pad, takes in (
            (8, 256, 256, 64, torch.bfloat16, 300, 0, False), (8, 256, 256, 128, torch.float32, 300, 0, False),
            (8, 256, 256, 128, torch.bfloat16, 300, 4, False), (8, 256, 256, 128, torch.bfloat16, 300, 0, True),
            (32, 256, 256, 128, torch.bfloat16, 20, 0, False),
            (8, 256, 256, 128, torch.bfloat16, 143, 0, False), (8, 256, 256, 128, torch.bfloat16, 144, 0, True),
            (4, 1024, 512, 128, torch.bfloat16, 35, 0, False), (4, 1024, 512, 128, torch.bfloat16, 36, 0, True),
            (64, 1024, 256, 128, torch.bfloat16, 511, 0, False), (64, 512, 256, 128, torch.bfloat16, 1024, 0, True),
            (8, 384, 384, 128, torch.bfloat16, 255, 0, False), (8, 384, 384, 128, torch.bfloat16, 256, 0, True),
            (4, 1024, 640, 128, torch.bfloat16, 114, 0, False), (4, 1024, 640, 128, torch.bfloat16, 115, 0, True)):
        bank = make_bank(experts, hidden, inter, group, torch.float32, gpu, 3)
        x = torch.randn(tokens, hidden + pad, device=gpu).to(dtype)[:, :hidden]
        logits = torch.randn(tokens, experts, device=gpu)
        assert takes_prefill(bank, x, logits, 2) == takes
        block = SparseMoeInt4(bank, num_experts=experts, top_k=2)
        assert rel_err(block(x, logits).double().cpu().numpy(), brute_force(bank, x, logits, 2, True)) <= BF16_TOL


def test_prefill_block_one_expert_past_a_million_routes(gpu):
    """87,500 chunks in 29,167 sweeps of one expert: the same bits as in calls of 100,000 tokens."""
    bank = make_bank(1, 128, 128, 128, torch.float32, gpu, 7)
    tokens = 1_400_000
    g = torch.Generator(device=gpu).manual_seed(9)
    x = torch.randn(tokens, 128, device=gpu, generator=g).to(torch.bfloat16)
    logits = torch.zeros(tokens, 1, device=gpu)
    block = SparseMoeInt4(bank, num_experts=1, top_k=1)
    got = block(x, logits)
    for a in range(0, tokens, 100_000):
        assert torch.equal(got[a:a + 100_000], block(x[a:a + 100_000], logits[a:a + 100_000]))


def test_unaligned_bank_takes_the_general_way(gpu):
    """Weights that are 4-byte aligned only (slices of one storage) give what aligned ones give."""
    bank = make_bank(16, 256, 256, 128, torch.float32, gpu, 11)
    torch.manual_seed(11)
    x = torch.randn(200, 256, device=gpu, dtype=torch.bfloat16)
    logits = torch.randn(200, 16, device=gpu)
    ref = brute_force(bank, x, logits, 4, True)
    for name in ("gate_qweight", "up_qweight", "down_qweight"):
        w = getattr(bank, name)
        room = torch.empty(w.numel() + 1, dtype=w.dtype, device=gpu)
        setattr(bank, name, room[1:].view(w.shape).copy_(w))
        assert not takes_prefill(bank, x, logits, 4)
        got = SparseMoeInt4(bank, num_experts=16, top_k=4)(x, logits)
        assert rel_err(got.double().cpu().numpy(), ref) <= BF16_TOL
