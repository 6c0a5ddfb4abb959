"""What is timed: the work a user of this framework has it do, through its public entry points.

Kinds of case
  linear    XPUInt4Linear.forward: one projection of a quantized layer (decode, batched decode, prefill)
  head      the quantized LM head and its top-k, one row for each sequence that samples a token
  moe       SparseMoeInt4: router, dispatch, grouped int4 MLP and combine of one sparse layer
  kv_decode one attention call of a decode step over a batched TurboQuant cache
  kv_load   prefill of every sequence of a batched TurboQuant cache, then the first decode step
  request   TurboQuantDynamicCache from empty: the prompt, then `steps` decode steps (append, attend)

Sizes are those of this repository's benchmark and tests (hidden 2048 and 4096, fused projections
of 6144 and 12288 rows, 128 experts with 8 per token, head_dim 128 and 256, 16 query heads on 2
key/value heads, a vocabulary of 151936) and, in draw(), the ranges around them.
"""

import math

import numpy as np
import torch

from anna_amd import fused_ops
from anna_amd.moe import GroupedInt4ExpertBank, SparseMoeInt4
from anna_amd.quantization import XPUInt4Linear
from anna_amd.tq_cache import TurboQuantBatchCache
from anna_amd.tq_dynamic import TurboQuantDynamicCache

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # one token through a projection: the smallest call, repeated for every layer and token
        dict(name="linear_m1", kind="linear", m=1, k=2048, n=6144, group=128, dtype="bf16", bias=False),
        # one decode step of a small batch through a fused gate/up projection
        dict(name="linear_m8", kind="linear", m=8, k=4096, n=12288, group=128, dtype="bf16", bias=False),
        # a short prompt of ragged length, with a bias, as an attention projection has
        dict(name="linear_m333_bias", kind="linear", m=333, k=4096, n=6144, group=128, dtype="bf16", bias=True),
        # a prefill chunk through the fused gate/up projection
        dict(name="linear_m2048", kind="linear", m=2048, k=4096, n=12288, group=128, dtype="bf16", bias=False),
        # sampling for a batch of four sequences from a large vocabulary
        dict(name="head_4rows", kind="head", rows=4, vocab=151936, k=2048, top_k=8, group=128, dtype="bf16"),
        # one decode step of eight sequences through a sparse layer
        dict(name="moe_decode", kind="moe", tokens=8, experts=128, top_k=8, hidden=2048, inter=512, group=128,
             dtype="bf16"),
        # a prefill chunk through the same layer
        dict(name="moe_prefill", kind="moe", tokens=2048, experts=128, top_k=8, hidden=2048, inter=512, group=128,
             dtype="bf16"),
        # attention of a decode step: long, unequal sequences, 2-bit cache
        dict(name="kv_decode_2bit", kind="kv_decode", batch=8, kv_heads=2, q_heads=16, head_dim=256, bits=2,
             mean_len=8704, gate=False),
        # the same on the 4-bit cache of a model with head_dim 128 and a gated output
        dict(name="kv_decode_4bit", kind="kv_decode", batch=8, kv_heads=2, q_heads=16, head_dim=128, bits=4,
             mean_len=8704, gate=True),
        # four prompts enter the 4-bit cache, and the first token after them
        dict(name="kv_load_4bit", kind="kv_load", batch=4, kv_heads=2, q_heads=16, head_dim=128, bits=4,
             mean_len=4096, gate=False),
        # a long prompt in the reference's key format, and a few tokens of answer
        dict(name="request_prompt", kind="request", batch=2, kv_heads=2, q_heads=16, head_dim=256, bits=4,
             prompt=8192, steps=4),
        # a short prompt and a longer answer for a batch
        dict(name="request_steps", kind="request", batch=8, kv_heads=2, q_heads=16, head_dim=128, bits=4,
             prompt=640, steps=24),
    ]


# ---------------------------------------------------------------- draw


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _size(rng, low, high, step):
    """A size of [low, high] over its logarithm: most often a multiple of `step`, now and then odd."""
    n = _log(rng, low, high)
    return max(low, min(high, n if rng.random() < 0.15 else -(-n // step) * step))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear", "head", "moe", "moe", "kv_decode", "kv_decode",
                       "kv_load", "request", "request"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    group = rng.choice([128, 128, 128, 64, 32])
    if kind == "linear":
        return dict(kind=kind, m=_log(rng, 1, 2048), k=_size(rng, 512, 4096, 256), n=_size(rng, 512, 12288, 128),
                    group=group, dtype=dtype, bias=rng.random() < 0.3)
    if kind == "head":
        return dict(kind=kind, rows=_log(rng, 1, 8), vocab=4 * _log(rng, 8000, 37984), k=rng.choice([1024, 2048]),
                    top_k=rng.choice([1, 8, 20]), group=128, dtype=dtype)
    if kind == "moe":
        return dict(kind=kind, tokens=_log(rng, 1, 2048), experts=rng.choice([32, 64, 128]), top_k=rng.choice([4, 8]),
                    hidden=rng.choice([1024, 2048]), inter=rng.choice([256, 512, 768]),
                    group=rng.choice([128, 128, 64]), dtype=dtype)
    kv_heads, groups = rng.choice([(2, 8), (4, 4), (8, 2), (2, 4), (4, 8)])
    head_dim, bits = rng.choice([(256, 2), (256, 2), (128, 4), (128, 2), (256, 4), (64, 4), (128, 3)])
    shape = dict(kv_heads=kv_heads, q_heads=kv_heads * groups, head_dim=head_dim, bits=bits)
    if kind == "request":
        # tokens of the whole prompt x heads x head_dim no more than the listed long prompt's
        batch = _log(rng, 1, 8)
        most = 2 * 8192 * 2 * 256 // (batch * kv_heads * head_dim)
        return dict(kind=kind, batch=batch, **shape, prompt=_log(rng, 32, min(8192, most)), steps=rng.randint(1, 12))
    batch = _log(rng, 1, 8)
    most = 8 * 8704 * 2 * 256 // (batch * kv_heads * head_dim) // (1 if kind == "kv_decode" else 4)
    return dict(kind=kind, batch=batch, **shape, mean_len=_log(rng, 160, min(16384, most)), gate=rng.random() < 0.5)


# ---------------------------------------------------------------- inputs


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _normal(g, *shape, dtype=torch.float32, scale=1.0):
    return (torch.randn(shape, device=DEVICE, generator=g) * scale).to(dtype)


def _int4(g, lead, n, k, group):
    """Codes, scales and zero points of `lead` stacked [n, k] weights as the quantizer leaves them:
    fp32 scales that make the rows of unit norm or so, zero points near the middle."""
    kp = -(-k // group) * group
    words = torch.randint(-(2**31), 2**31, (*lead, n, kp // 8), dtype=torch.int32, device=DEVICE, generator=g)
    shape = (*lead, kp // group, n)
    scales = (torch.rand(shape, device=DEVICE, generator=g) + 0.5) * (0.2 / math.sqrt(k))
    zeros = torch.randint(5, 11, shape, dtype=torch.int8, device=DEVICE, generator=g)
    return words, scales, zeros


def _linear_inputs(case, seed):
    g = _generator(seed)
    dtype = DTYPES[case["dtype"]]
    w = _int4(g, (), case["n"], case["k"], case["group"])
    bias = _normal(g, case["n"], dtype=dtype, scale=0.5) if case["bias"] else None
    return w, bias, _normal(g, case["m"], case["k"], dtype=dtype)


def _head_inputs(case, seed):
    g = _generator(seed)
    w = _int4(g, (), case["vocab"], case["k"], case["group"])
    return w, _normal(g, case["rows"], case["k"], dtype=DTYPES[case["dtype"]])


def _moe_inputs(case, seed):
    g = _generator(seed)
    e, h, i, group = case["experts"], case["hidden"], case["inter"], case["group"]
    gate, up, down = (_int4(g, (e,), n, k, group) for n, k in ((i, h), (i, h), (h, i)))
    x = _normal(g, case["tokens"], h, dtype=DTYPES[case["dtype"]])
    return gate, up, down, x, _normal(g, case["tokens"], e)


def _lengths(case):
    """Unequal sequence lengths with the case's mean: half of it to one and a half times it."""
    b, mean = case["batch"], case["mean_len"]
    return [mean] if b == 1 else [max(1, int(mean * (0.5 + i / (b - 1))) + i % 3) for i in range(b)]


def _keys_values(g, *shape):
    """Keys with a few strong channels, as rotary models have, and plain values."""
    channel = 1.0 + 3.0 * (torch.rand(shape[-1], device=DEVICE, generator=g) < 0.05)
    keys = (torch.randn(shape, device=DEVICE, generator=g) * channel).to(torch.bfloat16)
    return keys, torch.randn(shape, device=DEVICE, generator=g).to(torch.bfloat16)


def _kv_inputs(case, seed):
    g = _generator(seed)
    h, d = case["kv_heads"], case["head_dim"]
    rows = [_keys_values(g, h, n, d) for n in _lengths(case)]
    new = _keys_values(g, case["batch"], h, d)
    q = _normal(g, case["batch"], case["q_heads"], d, dtype=torch.bfloat16, scale=2.0)
    gate = _normal(g, case["batch"], case["q_heads"], d, dtype=torch.bfloat16) if case["gate"] else None
    return rows, new, q, gate


def _request_inputs(case, seed):
    g = _generator(seed)
    b, h, d = case["batch"], case["kv_heads"], case["head_dim"]
    prompt = _keys_values(g, b, h, case["prompt"], d)
    steps = [(*_keys_values(g, b, h, 1, d), _normal(g, b, case["q_heads"], 1, d, dtype=torch.bfloat16, scale=2.0))
             for _ in range(case["steps"])]
    return prompt, steps


# ---------------------------------------------------------------- prepare and run


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("linear", "head"):
        if kind == "linear":
            (words, scales, zeros), bias, x = _linear_inputs(case, seed)
        else:
            (words, scales, zeros), x = _head_inputs(case, seed)
            bias = None
        layer = XPUInt4Linear(x.shape[1], words.shape[0], group_size=case["group"], bias=bias is not None,
                              compute_dtype=x.dtype, device=DEVICE)
        with torch.no_grad():
            layer.qweight.copy_(words)
            layer.qscale.copy_(scales)
            layer.qzeros.copy_(zeros)
            if bias is not None:
                layer.bias.copy_(bias)
        if kind == "head":
            fused_ops.register_ops()
            layer.prepare_lm_head_topk_layout()
        return dict(case=case, layer=layer, x=x)
    if kind == "moe":
        gate, up, down, x, logits = _moe_inputs(case, seed)
        e = case["experts"]
        bank = GroupedInt4ExpertBank(e, case["hidden"], case["inter"], case["group"], *gate, *up, *down,
                                     slot_to_expert=list(range(e)), expert_to_slot={i: i for i in range(e)})
        return dict(case=case, block=SparseMoeInt4(bank, num_experts=e, top_k=case["top_k"]), x=x, logits=logits)
    scaling = 1.0 / math.sqrt(case["head_dim"])
    if kind == "request":
        prompt, steps = _request_inputs(case, seed)
        return dict(case=case, prompt=prompt, steps=steps, scaling=scaling)
    rows, new, q, gate = _kv_inputs(case, seed)
    cache = TurboQuantBatchCache(batch=case["batch"], kv_heads=case["kv_heads"], q_heads=case["q_heads"],
                                 capacities=[n + 64 for n in _lengths(case)], head_dim=case["head_dim"],
                                 bits=case["bits"], device=DEVICE)
    if kind == "kv_decode":
        for b, (k, v) in enumerate(rows):
            cache.load_sequence(b, k, v)
    return dict(case=case, cache=cache, rows=rows, new=new, q=q, gate=gate, scaling=scaling)


@torch.no_grad()
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        return state["layer"](state["x"])
    if kind == "head":
        layer = state["layer"]
        return torch.ops.anna.lm_head_int4_topk_fused(state["x"], *layer.lm_head_topk_tensors(), layer.group_size,
                                                      layer.in_features, case["top_k"])
    if kind == "moe":
        return state["block"](state["x"], state["logits"])
    if kind == "request":
        cache = TurboQuantDynamicCache(1, kv_cache_quant_bits=case["bits"])
        cache.update(*state["prompt"], 0, require_dense_cache=False)
        out = []
        for k, v, q in state["steps"]:
            cache.update(k, v, 0, require_dense_cache=False)
            out.append(cache.turboquant_single_token_decode_attention(
                0, q, scaling=state["scaling"], num_key_value_groups=case["q_heads"] // case["kv_heads"]))
        return out
    cache = state["cache"]
    if kind == "kv_load":
        for b, (k, v) in enumerate(state["rows"]):
            cache.load_sequence(b, k, v)
        cache.append(*state["new"])
    return cache.decode(state["q"], scaling=state["scaling"], gate=state["gate"])


# ---------------------------------------------------------------- work


def _packed_bytes(case, tokens):
    """Bytes of `tokens` cached tokens of one key/value head (the default window aside)."""
    d, bits = case["head_dim"], case["bits"]
    code = d * (2 if bits == 2 else 4) // 8
    if case["kind"] == "request":  # a byte for each index and each sign, two fp32 norms; min/max values
        return tokens * (2 * d + 8 + code + 4 * (d // 32))
    if (d, bits) == (256, 2):
        return tokens * 2 * (code + 2)
    return tokens * (2 * code + 2 + 4 * (d // 32))


def work(case):
    kind = case["kind"]
    if kind in ("linear", "head"):
        m, n, k = (case["m"], case["n"], case["k"]) if kind == "linear" else (case["rows"], case["vocab"], case["k"])
        kp = -(-k // case["group"]) * case["group"]
        out = 2 * m * n if kind == "linear" else m * case["top_k"] * 10
        return {"bytes": n * kp // 2 + kp // case["group"] * n * 5 + 2 * m * k + out, "flops": 2 * m * n * k}
    if kind == "moe":
        t, h, i, top = case["tokens"], case["hidden"], case["inter"], case["top_k"]
        routes = t * top
        active = case["experts"] * (1.0 - (1.0 - top / case["experts"]) ** t)  # experts with a route, on average
        weights = active * 3 * h * i * (0.5 + 5 / case["group"])
        return {"bytes": weights + 4 * t * h + 4 * t * case["experts"], "flops": 6 * routes * h * i}
    h, hq, d, window = case["kv_heads"], case["q_heads"], case["head_dim"], 128
    if kind == "request":
        b, n, steps = case["batch"], case["prompt"], case["steps"]
        read = b * h * 4 * d * (n + steps) + 4 * b * hq * d * steps
        packed = max(0, n + steps - window)
        written = b * h * _packed_bytes(case, packed) + b * h * 4 * d * min(window, n + steps)
        attended = sum(b * h * (_packed_bytes(case, max(0, n + s - window)) + 4 * d * min(window, n + s))
                       for s in range(1, steps + 1))
        flops = b * h * packed * 4 * d * d + sum(4 * b * hq * d * (n + s) for s in range(1, steps + 1))
        return {"bytes": read + written + attended, "flops": flops}
    cached, tokens, loaded = 0, 0, 0
    for n in _lengths(case):
        n += kind == "kv_load"
        cached += h * (_packed_bytes(case, max(0, n - window)) + 4 * d * min(window, n))
        tokens += n
        loaded += 4 * h * n * d
    both = cached + (loaded + cached if kind == "kv_load" else 0)
    return {"bytes": both + 4 * case["batch"] * hq * d, "flops": 4 * hq * d * tokens}


# ---------------------------------------------------------------- tolerance


def tolerance(case):
    # Sums are in fp32 and results are rounded to 16 bits (2^-9 and 2^-12 of the value at the most);
    # products of many rows round each weight to 16 bits as well, those of few do not.  Against 64
    # bits: projections are 1.6e-3 to 2.8e-3 off in bf16 and 2.1e-4 to 2.9e-4 in fp16, the sparse
    # block (which rounds its activations too, to bf16 for long prompts) 3.3e-3 and 1.7e-3, the
    # attention over a packed cache 1.7e-3 to 2.8e-3.  Allowed is about four times that.
    bf16 = case.get("dtype") == "bf16"
    if case["kind"] == "head":
        return {"rel": 8e-3 if bf16 else 1e-3, "differ": 1e-2}
    if case["kind"] == "linear":
        return {"rel": 1.1e-2 if bf16 else 1.2e-3}
    if case["kind"] == "moe":
        return {"rel": 1.3e-2 if bf16 else 7e-3}
    return {"rel": 1.1e-2}


# ---------------------------------------------------------------- the same in 64 bits


def _dequant(words, scales, zeros, k):
    """(code - zero) * scale in float64, [..., n, k]."""
    shifts = torch.arange(0, 32, 4, device=words.device, dtype=torch.int32)
    codes = ((words.unsqueeze(-1) >> shifts) & 15).flatten(-2).double()
    group = codes.shape[-1] // scales.shape[-2]
    s, z = (t.double().transpose(-1, -2).repeat_interleave(group, dim=-1) for t in (scales, zeros))
    return ((codes - z) * s)[..., :k]


def _splitmix64(seed, n):
    with np.errstate(over="ignore"):
        z = np.uint64(seed) + np.arange(1, n + 1, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return z ^ (z >> np.uint64(31))


def _rotation(d, seed=42):
    """The cache's seeded randomized Hadamard rotation, float64 [d, d]."""
    words = _splitmix64(seed, d // 64)
    bits = (words[:, None] >> np.arange(64, dtype=np.uint64)) & np.uint64(1)
    signs = 1.0 - 2.0 * bits.reshape(-1).astype(np.float64)
    had = np.ones((1, 1))
    while had.shape[0] < d:
        had = np.block([[had, had], [had, -had]])
    return torch.from_numpy(had * signs[None, :] / math.sqrt(d)).to(DEVICE)


def _gaussian(d, seed=42 ^ 0x514A4C):
    """The seeded normal matrix behind the sign sketch of the keys' residuals, float64 [d, d]."""
    u = ((_splitmix64(seed, d * d) >> np.uint64(11)).astype(np.float64) + 0.5) / 9007199254740992.0
    r, a = np.sqrt(-2.0 * np.log(u[0::2])), 2.0 * np.pi * u[1::2]
    g = np.stack([r * np.cos(a), r * np.sin(a)], axis=1).reshape(d, d)
    return torch.from_numpy(g.astype(np.float32).astype(np.float64)).to(DEVICE)


_LEVELS = {  # Lloyd-Max levels of a normal variable, the positive half
    1: [0.79788456080286629],
    2: [0.45278003463649735, 0.45278003463649735 * 3.74609375 / 1.123046875],
    3: [0.2450941789442308, 0.75600528120588584, 1.3439092785050075, 2.151945704536995],
    4: [0.12839502985114548, 0.38804829949029002, 0.65675911853246316, 0.94234045648696207, 1.2562311973471787,
        1.6180463860218879, 2.0690172265313875, 2.732589570995156],
}


def _levels(bits, d):
    half = torch.tensor(_LEVELS[bits], dtype=torch.float64, device=DEVICE) / math.sqrt(d)
    return torch.cat([-half.flip(0), half])


def _nearest(y, norm, levels):
    """The levels that the rotated vectors y of norm `norm` are coded to."""
    cuts = (levels[1:] + levels[:-1]) / 2
    return levels[torch.bucketize(y / norm.clamp_min(1e-300), cuts, right=True)]


def _mse(x, bits):
    """x as its rotated low-bit code and fp16 norm say it, float64 (last dimension: the vector)."""
    d = x.shape[-1]
    rot, x = _rotation(d), x.double()
    norm = x.norm(dim=-1, keepdim=True)
    return norm.half().double() * (_nearest(x @ rot.t(), norm, _levels(bits, d)) @ rot)


def _inner(x, bits):
    """x as bits - 1 bits of code and the sign sketch of the residual say it, in the cache's bf16."""
    d = x.shape[-1]
    rot, g, x = _rotation(d), _gaussian(d), x.double()
    norm = x.norm(dim=-1, keepdim=True)
    y = x @ rot.t()
    c = _nearest(y, norm, _levels(bits - 1, d))
    rho = y - c * norm
    signs = torch.where(rho @ g.t() >= 0, 1.0, -1.0).double()
    gamma = rho.norm(dim=-1, keepdim=True) / norm
    back = norm * ((c + math.sqrt(math.pi / 2) / d * gamma * (signs @ g)) @ rot)
    return back.to(torch.bfloat16).double()


def _minmax(x, bits, group=32):
    """x as min/max codes of groups with bf16 scales and zeros say it."""
    v = x.double().unflatten(-1, (-1, group))
    low, high = v.amin(-1, keepdim=True), v.amax(-1, keepdim=True)
    step = ((high - low) / (2**bits - 1)).clamp_min(1e-8).to(torch.bfloat16).double()
    return (((v - low) / step).round().clamp(0, 2**bits - 1) * step + low).flatten(-2)


def _attend(q, keys, values, scaling):
    """q [hq, d], keys and values [h, n, d] -> [hq, d], float64."""
    h = keys.shape[0]
    s = torch.matmul(q.double().reshape(h, -1, q.shape[-1]), keys.transpose(1, 2).contiguous()) * scaling
    return torch.matmul(torch.softmax(s, dim=-1), values).reshape(q.shape)


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        w, bias, x = _linear_inputs(case, seed)
        y = x.double() @ _dequant(*w, case["k"]).t()
        return y if bias is None else y + bias.double()
    if kind == "head":
        w, x = _head_inputs(case, seed)
        words, scales, zeros = w
        parts = [x.double() @ _dequant(words[i:i + 16384], scales[:, i:i + 16384], zeros[:, i:i + 16384], case["k"]).t()
                 for i in range(0, case["vocab"], 16384)]
        top = torch.topk(torch.cat(parts, dim=1), case["top_k"], dim=1)
        return top.values, top.indices
    if kind == "moe":
        gate, up, down, x, logits = _moe_inputs(case, seed)
        p, chosen = torch.topk(torch.softmax(logits.double(), dim=-1), case["top_k"], dim=-1)
        p = p / p.sum(dim=-1, keepdim=True)
        out = torch.zeros(x.shape, dtype=torch.float64, device=x.device)
        for e in range(case["experts"]):
            token, place = (chosen == e).nonzero(as_tuple=True)
            if not token.numel():
                continue
            wg, wu = (_dequant(*(t[e] for t in w), case["hidden"]) for w in (gate, up))
            wd = _dequant(*(t[e] for t in down), case["inter"])
            xe = x[token].double()
            act = torch.nn.functional.silu(xe @ wg.t()) * (xe @ wu.t())
            out.index_add_(0, token, (act @ wd.t()) * p[token, place].unsqueeze(1))
        return out
    scaling = 1.0 / math.sqrt(case["head_dim"])
    window, bits = 128, case["bits"]
    if kind == "request":
        prompt, steps = _request_inputs(case, seed)
        keys = torch.cat([prompt[0]] + [k for k, _, _ in steps], dim=2)
        values = torch.cat([prompt[1]] + [v for _, v, _ in steps], dim=2)
        coded_k, coded_v = _inner(keys, bits), _minmax(values, bits)
        out = []
        for i, (_, _, q) in enumerate(steps):
            n = case["prompt"] + i + 1
            old = max(0, n - window)
            out.append(torch.stack([
                _attend(q[b, :, 0], torch.cat([coded_k[b, :, :old], keys[b, :, old:n].double()], dim=1),
                        torch.cat([coded_v[b, :, :old], values[b, :, old:n].double()], dim=1), scaling)
                for b in range(case["batch"])]).unsqueeze(2))
        return out
    rows, new, q, gate = _kv_inputs(case, seed)
    out = []
    for b, (k, v) in enumerate(rows):
        if kind == "kv_load":
            k, v = (torch.cat([t, n[b].unsqueeze(1)], dim=1) for t, n in zip((k, v), new))
        old = max(0, k.shape[1] - window)
        coded_v = _mse(v[:, :old], bits) if (case["head_dim"], bits) == (256, 2) else _minmax(v[:, :old], bits)
        out.append(_attend(q[b], torch.cat([_mse(k[:, :old], bits), k[:, old:].double()], dim=1),
                           torch.cat([coded_v, v[:, old:].double()], dim=1), scaling))
    y = torch.stack(out)
    return y if gate is None else y * torch.sigmoid(gate.double())
