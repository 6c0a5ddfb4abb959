"""The host module (csrc/torch_host.cpp): what its functions take, what they leave to their Python callers,
and that both ways give the same result.

Every call is made twice: as it is, and with a module that takes nothing.  `Watched` notes whether the
module answered, so that a call that quietly changes sides fails here."""

import pytest
import torch

from anna_amd import _lib, fused_ops
from anna_amd.moe import SparseMoeInt4
from anna_amd.quantization import XPUInt4Linear
from anna_amd.tq_cache import TurboQuantBatchCache
from anna_amd.tq_dynamic import TurboQuantDynamicCache
from tests._util import BF16_TOL, rel_err
from tests.test_moe_gpu import make_bank

pytestmark = pytest.mark.gpu


class Watched:
    """The host module; `declines` names functions that take nothing.  answered: (name, took it)."""

    def __init__(self, module, declines=()):
        self.module, self.declines, self.answered = module, declines, []

    def __getattr__(self, name):
        def call(*args, **kwargs):
            out = None if name in self.declines else getattr(self.module, name)(*args, **kwargs)
            self.answered.append((name, out is not None))
            return out
        return call


@pytest.fixture
def both(gpu, monkeypatch):
    """both(fn, name, takes): fn() with and without the module's `name`, checked to be (not) taken."""
    module = _lib.host()

    def run(fn, name, takes=True):
        out = []
        for declines in ((), (name,)):
            watched = Watched(module, declines)
            monkeypatch.setattr(_lib, "_host", watched)
            out.append(fn())
            assert watched.answered == [(name, takes and not declines)]
        monkeypatch.setattr(_lib, "_host", module)
        return out

    return run


def make_linear(gpu, k, n, dtype, bias):
    torch.manual_seed(k + n)
    return XPUInt4Linear.from_linear(torch.nn.Linear(k, n, bias=bias), group_size=128, compute_dtype=dtype, device=gpu)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("bias", [False, True])
@torch.no_grad()
def test_linear(both, gpu, dtype, bias):
    layer = make_linear(gpu, 256, 96, dtype, bias)
    wide = torch.randn(7, 2, 320, device=gpu).to(dtype)
    x = wide[:, 0, :256]
    cases = [(x.contiguous(), True), (x, True), (x[:1], True), (x[0], True), (x.contiguous().view(7, 1, 256), True),
             (wide[..., :256], False),                                  # rows of a strided batch
             (x.t().contiguous().t(), False),                           # columns apart
             (x.to(torch.float64), False)]                              # another type
    for value, takes in cases:
        got, want = both(lambda: layer(value), "int4_linear", takes)
        assert got.dtype == value.dtype and got.shape == (*value.shape[:-1], 96)
        assert torch.equal(got, want)
    with pytest.raises(RuntimeError):
        layer(x[:1].expand(3, 256))  # rows on top of each other: refused by both


def test_linear_with_a_bias_that_needs_a_gradient(both, gpu):
    layer = make_linear(gpu, 256, 96, torch.bfloat16, True)
    layer.bias.requires_grad_(True)
    x = torch.randn(3, 256, device=gpu, dtype=torch.bfloat16)
    got, want = both(lambda: layer(x), "int4_linear", False)
    assert got.requires_grad and torch.equal(got, want)
    with torch.no_grad():
        got, _ = both(lambda: layer(x), "int4_linear", True)
    assert not got.requires_grad and torch.equal(got, want)


def test_gemv_op(both, gpu):
    layer = make_linear(gpu, 256, 96, torch.bfloat16, False)
    w = (layer.qweight, layer.qscale, layer.qzeros)
    x = torch.randn(5, 256, device=gpu, dtype=torch.bfloat16)
    for value, takes in ((x, True), (x.t().contiguous().t(), False)):
        got, want = both(lambda: fused_ops._xpu_int4_gemv_impl(value, *w, 128, 256), "int4_linear", takes)
        assert torch.equal(got, want)
    for bad in (x[:0], x[:, :128]):
        with pytest.raises(RuntimeError):
            fused_ops._xpu_int4_gemv_impl(bad, *w, 128, 256)


# decode (one launch routes it), a middle size, and a prompt, whose own form the Python way does not have
@pytest.mark.parametrize("tokens,experts,top_k,dtype,same_form", [
    (3, 16, 4, torch.bfloat16, True), (32, 32, 8, torch.float16, True), (9, 8, 2, torch.float32, True),
    (200, 16, 4, torch.float32, True), (200, 16, 4, torch.bfloat16, False),
])
def test_moe_block(both, gpu, tokens, experts, top_k, dtype, same_form):
    bank = make_bank(experts, 256, 256, 128, torch.float32, gpu, tokens)
    torch.manual_seed(tokens)
    block = SparseMoeInt4(bank, num_experts=experts, top_k=top_k)
    wide = torch.randn(tokens, 320, device=gpu).to(dtype)
    logits = torch.randn(tokens, experts, device=gpu)
    apart = wide[:, :256].t().contiguous().t()
    padded = torch.randn(tokens, experts + 3, device=gpu)[:, :experts].copy_(logits)
    outs = []
    for x, lg, takes in ((wide[:, :256], logits, True), (wide[:, :256].contiguous(), padded, True),
                         (apart, logits, False), (wide[:, :256], logits.t().contiguous().t(), False)):
        got, want = both(lambda: block(x, lg), "moe_block", takes)
        assert got.shape == (tokens, 256) and got.dtype == dtype
        if same_form or not takes:
            assert torch.equal(got, want)
        else:
            assert rel_err(got.double().cpu().numpy(), want.double().cpu().numpy()) <= BF16_TOL
        outs.append(want)
    assert all(torch.equal(o, outs[0]) for o in outs[1:])


@pytest.mark.parametrize("head_dim,bits,name", [(256, 2, "decode_pool"), (128, 4, "decode_rows")])
@pytest.mark.parametrize("gated", [False, True])
def test_batched_decode(both, gpu, head_dim, bits, name, gated):
    torch.manual_seed(head_dim)
    cache = TurboQuantBatchCache(batch=2, kv_heads=2, q_heads=8, capacities=[400, 400], head_dim=head_dim, bits=bits)
    for b, n in enumerate((300, 90)):
        cache.load_sequence(b, *(torch.randn(2, n, head_dim, device=gpu, dtype=torch.bfloat16) for _ in range(2)))
    q = torch.randn(2, 8, head_dim, device=gpu, dtype=torch.bfloat16)
    gate = torch.randn_like(q) if gated else None
    apart = torch.randn(2, 8, head_dim + 8, device=gpu, dtype=torch.bfloat16)[..., :head_dim].copy_(q)
    cache.decode(q, scaling=0.09, gate=gate)  # (the rows cache makes room for the partials: the caller's work)
    got, want = both(lambda: cache.decode(q, scaling=0.09, gate=gate), name)
    assert torch.equal(got, want)
    out = torch.zeros_like(q)
    assert both(lambda: cache.decode(q, scaling=0.09, gate=gate, out=out), name)[0] is out
    assert torch.equal(out, want)
    # a query whose heads are apart: the pool's module call leaves it, the rows' caller does not even ask
    again = cache.decode(apart, scaling=0.09, gate=gate)
    assert torch.equal(again, want)
    for bad in (q[:1], q[:, :4], q.float(), q[..., :64]):
        with pytest.raises((ValueError, RuntimeError)):
            cache.decode(bad, scaling=0.09)


@pytest.mark.parametrize("quantizer", ["ip", "mse"])
def test_dynamic_decode(both, gpu, quantizer):
    torch.manual_seed(4)
    cache = TurboQuantDynamicCache(1, kv_cache_residual_len=32, key_quantizer=quantizer)
    k, v = (torch.randn(3, 2, 150, 128, device=gpu, dtype=torch.bfloat16) for _ in range(2))
    cache.update(k, v, 0, require_dense_cache=False)
    q = torch.randn(3, 8, 1, 128, device=gpu, dtype=torch.bfloat16)
    wide = torch.randn(3, 8, 1, 256, device=gpu, dtype=torch.bfloat16)[..., :128].copy_(q)
    outs = []
    for query, gate in ((q, None), (wide, None), (q, torch.zeros_like(q))):
        got, want = both(lambda: cache.turboquant_single_token_decode_attention(
            0, query, scaling=0.09, num_key_value_groups=4, gate=gate), "decode_rows")
        assert torch.equal(got, want)
        outs.append(got)
    assert torch.equal(outs[0], outs[1])


def test_append_has_no_other_way(gpu, monkeypatch):
    """What the module does not take is refused, and the cache is as it was."""
    cache = TurboQuantDynamicCache(1, kv_cache_residual_len=32)
    k = torch.randn(1, 2, 40, 128, device=gpu, dtype=torch.bfloat16)
    cache.update(k, k, 0, require_dense_cache=False)
    module = _lib.host()
    monkeypatch.setattr(_lib, "_host", Watched(module, ("tq_store",)))
    with pytest.raises(RuntimeError, match="append"):
        cache.update(k, k, 0, require_dense_cache=False)
    monkeypatch.setattr(_lib, "_host", module)
    assert cache.layer_lengths == [[40]] and cache._slabs[0].seq_lengths.tolist() == [40]
    cache.update(k, k, 0, require_dense_cache=False)
    assert cache._slabs[0].seq_lengths.tolist() == [80]
