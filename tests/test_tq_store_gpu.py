"""The one-launch append of the dynamic cache (anna_mi_tq_store) against rows that quantize token by
token: codes, norms, signs, reconstruction, values, window and lengths, bit for bit.

The rows (TurboQuantKVRow) run the separate quantizers, which their own tests hold to the oracle.
"""

import pytest
import torch

from anna_amd.tq_cache import TurboQuantBatchCache
from anna_amd.tq_dynamic import TurboQuantDynamicCache
from anna_amd.turboquant import TurboQuantKVRow

pytestmark = pytest.mark.gpu


def same(a, b):
    a, b = a.contiguous(), b.contiguous()
    assert a.shape == b.shape and a.dtype == b.dtype
    assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def check_row(cache, b, row):
    slab, n = cache._slabs[0], row.quantized_length
    got = cache.turboquant_rows[0][b]
    assert (got.length, got.quantized_length) == (row.length, n)
    pairs = [("vdata", "_vdata"), ("vscales", "_vscales"), ("vzeros", "_vzeros"), ("knorms", "_knorms")]
    if slab.key_quantizer == "ip":
        pairs += [("kidx", "_kcodes"), ("kqjl", "_kqjl"), ("krn", "_krn"), ("kdense", "_kdense")]
    else:
        pairs += [("kcodes", "_kcodes")]
    if n:
        for mine, theirs in pairs:
            same(getattr(slab, mine)[b, :, :n], getattr(row, theirs)[:, :n])
    wk, wv = slab.window(b)
    same(wk, row._residual_keys)
    same(wv, row._residual_values)


# chunks that stay inside the window, fill it exactly, cross it from part full, wrap it more than
# once, and single tokens; 17 x 2 heads vectors end inside a tile of 16
PLANS = [(5, 27, 1, 1), (40, 1, 1), (3, 30, 200, 1, 77), (32, 1, 33, 64)]


@pytest.mark.parametrize("head_dim,bits,key_quantizer,dtype,group", [
    (64, 4, "ip", torch.bfloat16, None), (128, 3, "ip", torch.float16, 16), (256, 2, "ip", torch.bfloat16, None),
    (512, 4, "ip", torch.float32, 64), (1024, 4, "ip", torch.bfloat16, 512), (128, 4, "mse", torch.bfloat16, None),
    (256, 2, "mse", torch.float32, 4), (64, 3, "mse", torch.float16, 1), (192, 4, "mse", torch.bfloat16, None),
    (1024, 2, "mse", torch.bfloat16, 1024),
])
@pytest.mark.parametrize("plan", PLANS)
def test_store_matches_rows(gpu, head_dim, bits, key_quantizer, dtype, group, plan):
    torch.manual_seed(head_dim + bits)
    batch, heads, window = 3, 2, 32
    cache = TurboQuantDynamicCache(1, kv_cache_quant_bits=bits, kv_cache_residual_len=window,
                                   key_quantizer=key_quantizer, value_group_size=group)
    rows = [TurboQuantKVRow(bits=bits, residual_len=window, value_group_size=group, key_quantizer=key_quantizer)
            for _ in range(batch)]
    total = 0
    for i, t in enumerate(plan):
        # [B, T, H, D] transposed: strides of the attention's own layout
        k = torch.randn(batch, t, heads, head_dim, device=gpu).to(dtype).transpose(1, 2)
        v = torch.randn(batch, t, heads, head_dim, device=gpu).to(dtype).transpose(1, 2)
        _, _, past = cache.update(k, v, 0, require_dense_cache=False)
        assert past.dtype == torch.int64 and past.tolist() == [r.length for r in rows]
        for b in range(batch):
            rows[b].append(k[b], v[b])
        if i == 1:  # one sequence moves ahead of the others
            ek, ev = (torch.randn(heads, 7, head_dim, device=gpu).to(dtype) for _ in range(2))
            cache.append_row(0, 1, ek, ev)
            rows[1].append(ek, ev)
        total += t
        for b in range(batch):
            check_row(cache, b, rows[b])
        assert cache._slabs[0].seq_lengths.tolist() == [r.length for r in rows]


def test_large_tiles_match_small_ones(gpu):
    """A prompt long enough for the tiles of 64 vectors equals the same tokens in two chunks of the
    tiles of 16 (both end inside a tile)."""
    torch.manual_seed(3)
    for head_dim in (64, 128, 256, 512):
        k, v = (torch.randn(1, 2, 4321, head_dim, device=gpu, dtype=torch.bfloat16) for _ in range(2))
        caches = [TurboQuantDynamicCache(1, kv_cache_quant_bits=4) for _ in range(2)]
        caches[0].update(k, v, 0, require_dense_cache=False)
        for a, z in ((0, 3000), (3000, 4321)):
            caches[1].update(k[:, :, a:z], v[:, :, a:z], 0, require_dense_cache=False)
        one, two = (c._slabs[0] for c in caches)
        n = 4321 - 128
        for name in ("kidx", "knorms", "kqjl", "krn", "kdense", "vdata", "vscales", "vzeros"):
            same(getattr(one, name)[:, :, :n], getattr(two, name)[:, :, :n])
        same(one.rk, two.rk)
        same(one.rv, two.rv)


@pytest.mark.parametrize("head_dim,bits", [(128, 4), (64, 2), (512, 3)])
@pytest.mark.parametrize("length", [1, 128, 129, 700])
def test_rows_cache_load_equals_appends(gpu, head_dim, bits, length):
    """load_sequence over a row that held other tokens leaves what as many appends leave."""
    torch.manual_seed(length)
    batch, heads = 2, 2
    caches = [TurboQuantBatchCache(batch=batch, kv_heads=heads, q_heads=2 * heads, capacities=[640, 700],
                                   head_dim=head_dim, bits=bits) for _ in range(2)]
    k, v = (torch.randn(length, batch, heads, head_dim, device=gpu, dtype=torch.bfloat16) for _ in range(2))
    for t in range(length):
        caches[0].append(k[t], v[t])
    caches[1].load_sequence(1, *(torch.randn(heads, 300, head_dim, device=gpu, dtype=torch.bfloat16) for _ in range(2)))
    for b in range(batch):
        caches[1].load_sequence(b, k[:, b].transpose(0, 1), v[:, b].transpose(0, 1))
    one, two = caches
    assert one.lengths == two.lengths == one.seq_lengths.tolist() == two.seq_lengths.tolist()
    n, r = max(0, length - 128), min(length, 128)
    for name in ("key_codes", "key_norms", "value_data", "value_scales", "value_zeros"):
        same(getattr(one, name)[:, :, :n], getattr(two, name)[:, :, :n])
    for name in ("residual_key", "residual_value"):
        same(getattr(one, name)[:, :, :r], getattr(two, name)[:, :, :r])


def test_store_refusals(gpu):
    cache = TurboQuantDynamicCache(1, kv_cache_residual_len=16)
    good = torch.randn(2, 2, 20, 128, device=gpu, dtype=torch.bfloat16)
    cache.update(good, good, 0)
    with pytest.raises(RuntimeError):
        cache.update(good.cpu(), good.cpu(), 0)
    with pytest.raises(IndexError):
        cache.append_row(0, 2, good[0], good[0])
    # a head_dim the inner-product quantizer does not take is refused once tokens leave the window
    other = TurboQuantDynamicCache(1, kv_cache_residual_len=16)
    odd = torch.randn(1, 2, 12, 96, device=gpu, dtype=torch.bfloat16)
    other.update(odd, odd, 0, require_dense_cache=False)
    with pytest.raises(ValueError):
        other.update(odd, odd, 0, require_dense_cache=False)


@pytest.mark.parametrize("length", [1, 31, 64, 65, 190, 417])
@pytest.mark.parametrize("window", [32, 64])
def test_pool_load_equals_appends(gpu, length, window):
    """load_sequence of the 2-bit pool over a row that held other tokens leaves what as many appends
    leave, for separate and interleaved layouts of keys and values."""
    torch.manual_seed(length)
    batch, heads, D = 2, 3, 256
    caches = [TurboQuantBatchCache(batch=batch, kv_heads=heads, q_heads=2 * heads, capacities=[448, 450],
                                   residual_capacity=window) for _ in range(2)]
    k, v = (torch.randn(length, batch, heads, D, device=gpu, dtype=torch.bfloat16) for _ in range(2))
    for t in range(length):
        caches[0].append(k[t], v[t])
    caches[1].load_sequence(0, *(torch.randn(heads, 300, D, device=gpu, dtype=torch.bfloat16) for _ in range(2)))
    caches[1].load_sequence(0, k[:, 0].transpose(0, 1), v[:, 0].transpose(0, 1).contiguous())
    caches[1].load_sequence(1, k[:, 1].transpose(0, 1), v[:, 1].transpose(0, 1))
    one, two = caches
    assert one.lengths == two.lengths == one.seq_lengths.tolist() == two.seq_lengths.tolist()
    q, r = max(0, length - window), min(length, window)
    for b in range(batch):
        s = slice(one.offsets[b], one.offsets[b] + q)
        for name in ("key_codes", "key_norms", "value_norms"):
            same(getattr(one, name)[:, s], getattr(two, name)[:, s])
        whole = slice(one.offsets[b] // 32, (one.offsets[b] + q // 32 * 32) // 32)  # blocks of 32 slots
        same(one.value_codes[:, whole], two.value_codes[:, whole])
    same(one.residual_key[:, :, :r], two.residual_key[:, :, :r])
    same(one.residual_value_t[..., :r], two.residual_value_t[..., :r])
    query = torch.randn(batch, 2 * heads, D, device=gpu, dtype=torch.bfloat16)
    same(one.decode(query, scaling=0.06), two.decode(query, scaling=0.06))


@pytest.mark.parametrize("quantizer", ["ip", "mse"])
def test_captured_decode_follows_the_appends(gpu, quantizer):
    """A decode captured in a graph reads the lengths of the replay: tokens appended between replays count,
    whether to every sequence or to one."""
    torch.manual_seed(8)
    head_dim = 128
    cache = TurboQuantDynamicCache(1, kv_cache_residual_len=16, key_quantizer=quantizer)
    new = lambda *s: torch.randn(*s, head_dim, device=gpu, dtype=torch.bfloat16)
    k, v = new(2, 2, 40), new(2, 2, 40)
    cache.update(k, v, 0, require_dense_cache=False)
    k, v = new(2, 2, 1), new(2, 2, 1)
    cache.update(k, v, 0, require_dense_cache=False)  # the slab has room from here on
    q = new(2, 4, 1)
    call = lambda: cache.turboquant_single_token_decode_attention(0, q, scaling=0.1, num_key_value_groups=2)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        call()
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    lengths = cache._slabs[0].seq_lengths
    for step in range(5):
        if step == 2:
            cache.append_row(0, 1, *(new(2, 3) for _ in range(2)))
        elif step:
            cache.update(new(2, 2, 1), new(2, 2, 1), 0, require_dense_cache=False)
        graph.replay()
        same(out, call())
        assert cache._slabs[0].seq_lengths is lengths and lengths.tolist() == cache.layer_lengths[0]


def odd_strides(t):
    """t with a stride of 1 in each dimension of size 1: contiguous to torch, whose rule skips those"""
    out = t.clone(memory_format=torch.contiguous_format)
    return out.as_strided(t.shape, [1 if n == 1 else s for n, s in zip(t.shape, out.stride())])


@pytest.mark.parametrize("batch,heads,tokens", [(3, 2, 1), (1, 2, 1), (1, 2, 40), (2, 1, 9), (1, 1, 1), (1, 1, 40)])
@pytest.mark.parametrize("key_quantizer", ["ip", "mse"])
def test_store_takes_any_stride_of_a_single_row(gpu, batch, heads, tokens, key_quantizer):
    torch.manual_seed(tokens)
    caches = [TurboQuantDynamicCache(1, kv_cache_residual_len=16, key_quantizer=key_quantizer) for _ in range(2)]
    for n in (tokens, 20, tokens):
        k, v = (torch.randn(batch, heads, n, 128, device=gpu, dtype=torch.bfloat16) for _ in range(2))
        caches[0].update(k, v, 0, require_dense_cache=False)
        caches[1].update(odd_strides(k), odd_strides(v), 0, require_dense_cache=False)
    for (ak, av), (bk, bv) in zip(*([r.materialize() for r in c.turboquant_rows[0]] for c in caches)):
        same(ak, bk)
        same(av, bv)


@pytest.mark.parametrize("head_dim,bits", [(128, 4), (256, 2)])
@pytest.mark.parametrize("heads,length", [(2, 1), (1, 1), (1, 150), (2, 150)])
def test_load_takes_any_stride_of_a_single_row(gpu, head_dim, bits, heads, length):
    torch.manual_seed(length)
    k, v = (torch.randn(heads, length, head_dim, device=gpu, dtype=torch.bfloat16) for _ in range(2))
    q = torch.randn(1, 2 * heads, head_dim, device=gpu, dtype=torch.bfloat16)
    out = []
    for a, b in ((k, v), (odd_strides(k), odd_strides(v)), (odd_strides(k), v), (k, odd_strides(v))):
        cache = TurboQuantBatchCache(batch=1, kv_heads=heads, q_heads=2 * heads, capacities=[64], head_dim=head_dim,
                                     bits=bits)
        cache.load_sequence(0, a, b)
        out.append(cache.decode(q, scaling=0.09))
    for o in out[1:]:
        same(o, out[0])
    # a token stride that no row of 8 bytes fits, of one token: nothing is read at it
    wide = torch.empty(heads * (head_dim + 1), device=gpu, dtype=torch.bfloat16)[:heads * head_dim]
    one = wide.view(heads, 1, head_dim).as_strided((heads, 1, head_dim), (head_dim, head_dim + 1, 1)).copy_(k[:, :1])
    cache.load_sequence(0, one, one)
    first = cache.decode(q, scaling=0.09)
    cache.load_sequence(0, k[:, :1], k[:, :1])
    same(first, cache.decode(q, scaling=0.09))


def test_load_of_nothing_and_of_other_types(gpu):
    """No tokens: any head_dim, and in the 2-bit pool any type, as there is nothing to read."""
    for head_dim, bits in ((256, 2), (128, 4)):
        cache = TurboQuantBatchCache(batch=1, kv_heads=2, q_heads=4, capacities=[64], head_dim=head_dim, bits=bits)
        k = torch.randn(2, 5, head_dim, device=gpu, dtype=torch.bfloat16)
        cache.load_sequence(0, k, k)
        if bits == 2:
            cache.load_sequence(0, k[:, :0].float(), k[:, :0].float())
        cache.load_sequence(0, k[:, :0, :64], k[:, :0, :64])
        assert cache.lengths == [0] == cache.seq_lengths.tolist()
        long = torch.randn(2, 150, head_dim, device=gpu, dtype=torch.bfloat16)
        for bad in (k.float(), k[..., :64], long[..., :64], long[..., :1]):
            with pytest.raises((ValueError, RuntimeError)):
                cache.load_sequence(0, bad, bad)
        # within the window a head, a token or a dimension of size 1 stands for all of them
        q = torch.randn(1, 4, head_dim, device=gpu, dtype=torch.bfloat16)
        for part in (k[:1], k[..., :1]):
            cache.load_sequence(0, part, part)
            got = cache.decode(q, scaling=0.09)
            cache.load_sequence(0, part.expand_as(k).contiguous(), part.expand_as(k).contiguous())
            same(got, cache.decode(q, scaling=0.09))


def test_value_groups_matter_once_tokens_leave(gpu):
    """A group size that does not divide head_dim is refused where a token is quantized, not before."""
    cache = TurboQuantDynamicCache(1, kv_cache_residual_len=16, value_group_size=48)
    k = torch.randn(2, 2, 16, 128, device=gpu, dtype=torch.bfloat16)
    keys, values, _ = cache.update(k, k, 0)
    same(keys, k)
    same(values, k)
    with pytest.raises((ValueError, RuntimeError)):
        cache.update(k, k, 0)


def test_update_of_no_sequences(gpu):
    cache = TurboQuantDynamicCache(1, kv_cache_residual_len=16)
    k = torch.randn(0, 2, 20, 128, device=gpu, dtype=torch.bfloat16)
    _, _, past = cache.update(k, k, 0, require_dense_cache=False)
    assert past.numel() == 0


def test_update_is_refused_in_a_capture(gpu):
    """The host counts the lengths and the append's arrays alternate, so that a replay would store the
    captured step again; a refused update leaves the cache as it was."""
    cache = TurboQuantDynamicCache(1, kv_cache_residual_len=16)
    k = torch.randn(2, 2, 20, 128, device=gpu, dtype=torch.bfloat16)
    cache.update(k, k, 0, require_dense_cache=False)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        one = k[:, :, :1] + 0
        with pytest.raises(RuntimeError, match="captured"):
            cache.update(one, one, 0, require_dense_cache=False)
    assert cache.layer_lengths == [[20, 20]]
    cache.update(k[:, :, :1], k[:, :, :1], 0, require_dense_cache=False)
    assert cache._slabs[0].seq_lengths.tolist() == [21, 21]
