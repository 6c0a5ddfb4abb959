"""int4 linear for groups of 32 or 64 and unaligned activations (int4_rows.hip) against sums in 64 bits."""

import pytest
import torch

from anna_amd import fused_ops

pytestmark = pytest.mark.gpu


def _payload(g, n, k, group, sdt):
    kp = -(-k // group) * group
    qw = torch.randint(-(2**31), 2**31, (n, kp // 8), dtype=torch.int32, generator=g)
    qs = ((torch.rand((kp // group, n), generator=g) + 0.5) * 0.05).to(sdt)
    qz = torch.randint(0, 16, (kp // group, n), dtype=torch.int8, generator=g)
    qz[0, : min(n, 4)] = torch.tensor([-128, -113, -112, 127], dtype=torch.int8)[: min(n, 4)]
    return qw, qs, qz


def _weight(qw, qs, qz, k, group):
    q = torch.stack([(qw >> (4 * j)) & 15 for j in range(8)], dim=-1).reshape(qw.shape[0], -1)
    idx = torch.arange(q.shape[1]) // group
    return ((q - qz.t().int()[:, idx]).double() * qs.t().double()[:, idx])[:, :k]


CASES = [
    # (M, K, N, group, row stride - K, scale dtype)
    (1, 512, 96, 32, 0, torch.float32),
    (1, 2048, 8200, 64, 0, torch.bfloat16),   # two tiles a workgroup, N tail
    (3, 1000, 50, 32, 0, torch.float32),      # K ends inside a block
    (8, 4096, 72, 64, 8, torch.float16),      # several blocks a wave, strided rows
    (16, 2944, 33, 64, 0, torch.float32),     # an odd number of blocks
    (17, 640, 100, 32, 0, torch.float32),     # two row groups
    (33, 1120, 40, 32, 0, torch.bfloat16),    # four row groups, the last empty
    (130, 1056, 70, 32, 0, torch.float32),    # three workgroups of rows
    (70, 232, 40, 64, 0, torch.float32),      # group 64 with K no multiple of 64
    (1, 333, 40, 128, 0, torch.float32),      # odd K: unaligned rows
    (5, 1237, 64, 128, 0, torch.bfloat16),
    (40, 1001, 48, 32, 3, torch.float32),     # odd K and row stride
    (200, 129, 20, 64, 0, torch.float32),
    (2, 1, 5, 128, 0, torch.float32),         # the smallest K
    # more than 512 pairs of a 16-row tile of W and a 16-row group of x: two tiles a workgroup
    (16, 320, 8200, 32, 0, torch.float32),
    (17, 640, 4113, 32, 0, torch.float32),    # and two row groups
    (33, 1120, 2801, 32, 0, torch.bfloat16),  # four row groups, the last empty
    (130, 1056, 930, 64, 0, torch.float32),   # three workgroups of rows
    (70, 232, 1700, 64, 0, torch.float32),    # group 64 with K no multiple of 64
    (40, 1001, 2800, 32, 3, torch.float32),   # odd K and row stride
    (200, 129, 640, 128, 0, torch.float16),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,k,n,group,pad,sdt", CASES)
def test_rows_against_64_bits(gpu, m, k, n, group, pad, sdt, dtype):
    print(f"[case] int4 rows M={m} K={k} N={n} g={group} pad={pad}", flush=True)
    g = torch.Generator().manual_seed(m * 31 + k + n)
    qw, qs, qz = _payload(g, n, k, group, sdt)
    x = torch.randn((m, k + pad), generator=g).to(dtype)
    w = _weight(qw, qs, qz, k, group)
    ref = x[:, :k].double() @ w.t()
    out = torch.empty((m, n), dtype=dtype, device=gpu)
    fused_ops.int4_linear_out(x.to(gpu)[:, :k], qw.to(gpu), qs.to(gpu), qz.to(gpu), group, k, out)
    # half a unit of the result's last place, and fp32 sums of k products (one more rounding for each scale)
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    bound = ref.abs() * unit + (x[:, :k].double().abs() @ w.abs().t()) * (k + 8) * 2.0 ** -24 + 2.0 ** -24
    assert bool(((out.cpu().double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("m", [1, 20])
def test_rows_keep_infinities(gpu, m):
    """An infinite activation reaches only its own row, as a signed infinity (NaN where q = z)."""
    g = torch.Generator().manual_seed(5)
    k, n, group = 256, 48, 32
    qw, qs, qz = _payload(g, n, k, group, torch.float32)
    x = torch.randn((m, k), generator=g).to(torch.bfloat16)
    x[0, 77] = float("inf")
    w = _weight(qw, qs, qz, k, group)
    out = torch.empty((m, n), dtype=torch.bfloat16, device=gpu)
    fused_ops.int4_linear_out(x.to(gpu), qw.to(gpu), qs.to(gpu), qz.to(gpu), group, k, out)
    want = w[:, 77] * float("inf")
    torch.testing.assert_close(out[0].cpu().double(), want, equal_nan=True)
    assert bool(torch.isfinite(out[1:]).all())


@pytest.mark.parametrize("m,n,k", [(193, 8832, 256), (385, 6000, 512)])
def test_gemm_middle_tile_past_a_round_of_small_tiles(gpu, monkeypatch, m, n, k):
    """More than 512 small tiles on less than a round of middle ones: the middle tile with K split."""
    monkeypatch.delenv("ANNA_MI_INT4_GEMM_TILE", raising=False)
    g = torch.Generator().manual_seed(m)
    qw, qs, qz = _payload(g, n, k, 128, torch.float32)
    qz.clamp_(0, 15)
    x = torch.randn((m, k), generator=g).to(torch.bfloat16)
    w = _weight(qw, qs, qz, k, 128)
    ref = x.double() @ w.t()
    out = torch.empty((m, n), dtype=torch.bfloat16, device=gpu)
    fused_ops.int4_linear_out(x.to(gpu), qw.to(gpu), qs.to(gpu), qz.to(gpu), 128, k, out)
    # W rounded to bf16 and the result: 2^-9 each of their magnitudes
    bound = ref.abs() * 2.0 ** -8 + (x.double().abs() @ w.abs().t()) * (2.0 ** -9 + (k + 8) * 2.0 ** -24)
    assert bool(((out.cpu().double() - ref).abs() <= bound).all())
