"""Tiled int4 GEMV (xpu_int4_gemv_tiled) and the fused int4 LM-head top-k against the CPU
dequant path.  Shapes follow the reference's tests (test_fused_op_xpu.py:260-375): indices
exact, values within the reference's 2e-2; the GEMV within normwise relative error 1e-2."""

import pytest
import torch

from anna_amd import fused_ops
from anna_amd.quantization import XPUInt4Linear
from oracle import cpu_paths as cp
from tests._util import BF16_TOL, rel_err

pytestmark = pytest.mark.gpu


def quantized_linear(k, n, seed, device, group=32, dtype=torch.float16):
    torch.manual_seed(seed)
    dense = torch.nn.Linear(k, n, bias=False, dtype=torch.float32)
    return XPUInt4Linear.from_linear(dense, group_size=group, compute_dtype=dtype, device=device)


def dense_logits(q, x):
    w = cp.int4_dequant_f32(q.qweight.cpu(), q.qscale.cpu(), q.qzeros.cpu(), q.group_size, q.in_features)
    return x.cpu().double() @ w.double().t()


@pytest.mark.parametrize("k,n,seed,layout", [(16, 31, 0, "plain"), (64, 96, 8, "lm_head"), (96, 192, 5, "plain"),
                                             (2048, 1000, 3, "lm_head"),
                                             (128, 20000, 4, "lm_head"),    # rows split over chunks (V >= 8192)
                                             (64, 8193, 6, "plain")])
def test_lm_head_int4_topk_matches_quantized_reference(gpu, k, n, seed, layout):
    q = quantized_linear(k, n, seed, gpu)
    x = torch.randn(2, 3, k, device=gpu, dtype=torch.float16)
    if layout == "lm_head":
        q.prepare_lm_head_topk_layout()
        tensors = (q.lm_head_qweight, q.lm_head_qscale, q.lm_head_qzeros)
    else:
        tensors = (q.qweight, q.qscale, q.qzeros)
    values, indices = torch.ops.anna.lm_head_int4_topk_fused(x, *tensors, q.group_size, q.in_features, 5)
    assert values.shape == (2, 3, 5) and indices.dtype == torch.long
    ref = dense_logits(q, x.reshape(-1, k)).view(2, 3, n)
    rv, ri = torch.topk(ref, 5, dim=-1)
    assert torch.equal(indices.cpu(), ri)
    torch.testing.assert_close(values.cpu().double(), rv, atol=2e-2, rtol=2e-2)
    # the module forward picks the same top-k
    mv, mi = torch.topk(q(x), 5, dim=-1)
    assert torch.equal(indices, mi)


@pytest.mark.parametrize("k,n,seed,layout,rows", [(2048, 1000, 13, "lm_head", 1), (2048, 4096, 14, "lm_head", 4),
                                                  (128, 20000, 15, "lm_head", 1), (200, 300, 16, "plain", 3),
                                                  (64, 8193, 17, "plain", 2)])
def test_lm_head_topk_few_rows(gpu, k, n, seed, layout, rows):
    """One to four rows: the tiled GEMV's LDS-staged form (x and the tiles' scales and zero
    points staged once per workgroup); K = 200 leaves the staged x rows unaligned to 4 words."""
    q = quantized_linear(k, n, seed, gpu, group=32)
    x = torch.randn(rows, k, device=gpu, dtype=torch.float16)
    if layout == "lm_head":
        q.prepare_lm_head_topk_layout()
        tensors = (q.lm_head_qweight, q.lm_head_qscale, q.lm_head_qzeros)
    else:
        tensors = (q.qweight, q.qscale, q.qzeros)
    values, indices = torch.ops.anna.lm_head_int4_topk_fused(x, *tensors, q.group_size, q.in_features, 6)
    ref = dense_logits(q, x)
    rv, ri = torch.topk(ref, 6, dim=-1)
    assert torch.equal(indices.cpu(), ri)
    torch.testing.assert_close(values.cpu().double(), rv, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("tile,sdt,m,k,group", [(1, torch.float32, 1, 256, 64), (2, torch.bfloat16, 3, 256, 64),
                                                (4, torch.float16, 5, 256, 64), (8, torch.float32, 2, 256, 64),
                                                (4, torch.bfloat16, 4, 200, 32), (8, torch.bfloat16, 1, 4096, 128)])
def test_xpu_int4_gemv_tiled_matches_dequant(gpu, tile, sdt, m, k, group):
    q = quantized_linear(k, 200, 11 + tile, gpu, group=group, dtype=torch.bfloat16)
    n, pc = q.qweight.shape
    n_pad = -(-n // tile) * tile
    qw = torch.zeros((n_pad, pc), dtype=torch.int32, device=gpu)
    qw[:n] = q.qweight
    qs = torch.ones((q.qscale.shape[0], n_pad), dtype=sdt, device=gpu)
    qs[:, :n] = q.qscale.to(sdt)
    qz = torch.full((q.qzeros.shape[0], n_pad), 8, dtype=torch.int8, device=gpu)
    qz[:, :n] = q.qzeros
    qw_t = qw.view(n_pad // tile, tile, pc).permute(0, 2, 1).contiguous()
    x = torch.randn(m, k, device=gpu, dtype=torch.bfloat16)
    y = torch.ops.anna.xpu_int4_gemv_tiled(x, qw_t, qs.view(-1, n_pad // tile, tile), qz.view(-1, n_pad // tile, tile),
                                           group, k, n)
    assert y.shape == (m, n) and y.dtype == torch.bfloat16
    w = cp.int4_dequant_f32(q.qweight.cpu(), q.qscale.to(sdt).cpu(), q.qzeros.cpu(), group, k)
    ref = x.cpu().double() @ w.double().t()
    assert rel_err(y.cpu().double().numpy(), ref.numpy()) <= BF16_TOL


def test_lm_head_topk_errors(gpu):
    q = quantized_linear(16, 31, 0, gpu)
    x = torch.randn(1, 16, device=gpu, dtype=torch.float16)
    with pytest.raises(RuntimeError, match="top_k"):
        fused_ops.run_lm_head_int4_topk_fused(hidden_states=x, qweight=q.qweight, qscale=q.qscale, qzeros=q.qzeros,
                                              group_size=32, in_features=16, top_k=40)
    with pytest.raises(RuntimeError, match="in_features"):
        fused_ops.run_lm_head_int4_topk_fused(hidden_states=x, qweight=q.qweight, qscale=q.qscale, qzeros=q.qzeros,
                                              group_size=32, in_features=8, top_k=3)


@pytest.mark.parametrize("v,rows,k", [(31, 1, 5), (5000, 3, 8), (20000, 2, 16), (3000, 1, 32), (40, 2, 32)])
def test_topk_rows_exact_with_ties(gpu, v, rows, k):
    """The row top-k (both kernels: k <= 8 in registers, k > 8 in LDS) against a CPU sort by
    (value descending, index ascending), with many exact ties."""
    from anna_amd import _lib
    print(f"[case] topk_rows V={v} rows={rows} k={k}", flush=True)
    g = torch.Generator().manual_seed(v + k)
    vals = torch.randn(rows, v, generator=g)
    vals[:, ::7] = vals[:, :1]  # every 7th value ties with the first
    dev_vals = vals.to(gpu)
    out_v = torch.empty((rows, k), dtype=torch.float32, device=gpu)
    out_i = torch.empty((rows, k), dtype=torch.int64, device=gpu)
    _lib.call("anna_mi_topk_rows", dev_vals.data_ptr(), rows, v, v, k, out_v.data_ptr(), _lib.dtype_code(torch.float32),
              out_i.data_ptr(), _lib.stream_of(dev_vals))
    for r in range(rows):
        order = sorted(range(v), key=lambda i: (-float(vals[r, i]), i))[:k]
        assert out_i[r].cpu().tolist() == order
        assert torch.equal(out_v[r].cpu(), vals[r, order])


@pytest.mark.parametrize("layout", ["lm_head", "plain"])
def test_lm_head_topk_exact_ties_in_wave_path(gpu, layout):
    """Few long rows take the wave-level top-k (chunk lists and a head tournament across lanes):
    with every weight row duplicated 6144 rows later, each logit ties exactly with its twin, and
    the pairs must come out value-descending, lower index first."""
    torch.manual_seed(99)
    dense = torch.nn.Linear(256, 12288, bias=False, dtype=torch.float32)
    with torch.no_grad():
        dense.weight[6144:] = dense.weight[:6144]
    q = XPUInt4Linear.from_linear(dense, group_size=32, compute_dtype=torch.float16, device=gpu)
    x = torch.randn(2, 256, device=gpu, dtype=torch.float16)
    if layout == "lm_head":
        q.prepare_lm_head_topk_layout()
        tensors = (q.lm_head_qweight, q.lm_head_qscale, q.lm_head_qzeros)
    else:
        tensors = (q.qweight, q.qscale, q.qzeros)
    values, indices = torch.ops.anna.lm_head_int4_topk_fused(x, *tensors, q.group_size, q.in_features, 8)
    ref = dense_logits(q, x)
    for r in range(2):
        order = sorted(range(12288), key=lambda i: (-float(ref[r, i]), i))[:8]
        assert indices[r].cpu().tolist() == order
        got = values[r].float().cpu()
        assert torch.equal(got[0::2], got[1::2])  # twins carry the same value


@pytest.mark.parametrize("k,n,rows,top_k,dtype,group", [
    (128, 8192, 1, 1, torch.bfloat16, 128), (256, 8196, 2, 8, torch.float16, 128), (512, 9000, 3, 32, torch.bfloat16, 128),
    (640, 16444, 5, 20, torch.float16, 128), (1024, 70004, 9, 8, torch.bfloat16, 256),
    (2048, 12300, 17, 9, torch.bfloat16, 128), (2176, 8260, 33, 5, torch.float16, 128),
    (512, 49996, 1, 8, torch.bfloat16, 128), (512, 50000, 1, 8, torch.bfloat16, 128), (512, 50000, 1, 9, torch.float16, 128),
    (2560, 50000, 1, 3, torch.float16, 128), (2432, 12284, 2, 3, torch.float16, 128), (2432, 12288, 2, 3, torch.bfloat16, 128),
])
def test_lm_head_block_selection(gpu, k, n, rows, top_k, dtype, group):
    """Whole 128-k blocks on tiles of 4 rows: the MFMA GEMV (K short of four waves' shares, ragged last
    block of rows, one to three 16-row blocks of x) and the selection over 64-logit blocks, and the shapes that
    take the GEMV and the chunk lists instead, against fp64;
    repeated weight rows make exact ties, which go to the lower index."""
    torch.manual_seed(k + n)
    kp = -(-k // group) * group
    q = XPUInt4Linear(k, n, group_size=group, compute_dtype=dtype, device=gpu)
    with torch.no_grad():
        q.qweight.copy_(torch.randint(-(2**31), 2**31, (n, kp // 8), dtype=torch.int32, device=gpu))
        q.qscale.copy_(torch.rand(kp // group, n, device=gpu) * 0.01 + 0.001)
        q.qzeros.copy_(torch.randint(-128, 128, (kp // group, n), dtype=torch.int8, device=gpu))
        for buf, dim in ((q.qweight, 0), (q.qscale, 1), (q.qzeros, 1)):  # the last 70 rows repeat the first 70
            buf.narrow(dim, n - 70, 70).copy_(buf.narrow(dim, 0, 70))
    q.prepare_lm_head_topk_layout()
    x = torch.randn(rows, k, device=gpu, dtype=dtype)
    values, indices = torch.ops.anna.lm_head_int4_topk_fused(x, q.lm_head_qweight, q.lm_head_qscale, q.lm_head_qzeros,
                                                             group, k, top_k)
    ref = dense_logits(q, x).to(gpu)
    rv, _ = torch.topk(ref, top_k, dim=-1)
    # fp32 sums of up to 2176 products of |code - zero| <= 143 against values of a few hundred, then the
    # output's rounding (2^-9 or 2^-12 of the value)
    eps = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-10
    scale = ref.abs().amax()
    assert ((values.double() - rv).abs() <= eps * rv.abs() + 1e-5 * scale).all()
    assert ((torch.gather(ref, 1, indices) - rv).abs() <= 1e-5 * scale).all()
    assert all(len(set(r.tolist())) == top_k for r in indices)
    for row in indices.tolist():  # a repeated row never stands before the row it repeats
        for place, i in enumerate(row):
            if i >= n - 70:
                assert i - (n - 70) in row[:place]
    # the GEMV alone, in the activation dtype
    y = fused_ops.int4_gemv_tiled(x, q.lm_head_qweight, q.qscale.view(-1, n // 4, 4), q.qzeros.view(-1, n // 4, 4),
                                  group, k, n)
    assert rel_err(y.double().cpu().numpy(), ref.cpu().numpy()) <= BF16_TOL


@pytest.mark.parametrize("m,n,k", [(1, 24576, 128), (1, 24580, 128), (4, 1536, 256), (4, 1540, 256), (5, 300, 256),
                                   (5, 3932, 512), (5, 3936, 512), (1, 32768, 512), (1, 32772, 512), (6, 300, 512),
                                   (4, 6144, 768), (4, 6148, 768), (5, 300, 768), (2, 6144, 1152), (2, 6148, 1536),
                                   (3, 300, 2048), (3, 2728, 4096), (3, 2732, 4096), (2, 2048, 4224), (2, 2052, 4224), (3, 300, 4224),
                                   (6, 6144, 512), (6, 6148, 512), (2, 55296, 384), (2, 55300, 384), (5, 3936, 768),
                                   (6, 300, 768), (4, 6144, 1536), (4, 6148, 1536), (1, 50000, 1536), (3, 5460, 2048),
                                   (3, 5464, 2048), (4, 300, 2048), (4, 4096, 2176), (4, 4096, 4096), (4, 4100, 4096), (1, 24580, 2048), (4, 6144, 4224), (4, 6148, 4224),
                                   (1, 12288, 4224), (1, 12292, 4224)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_tiled_gemv_on_both_sides_of_its_forms(gpu, m, n, k, dtype):
    """Tiles of 4 rows and whole 128-k blocks: the dot2 forms for few rows, the MFMA form beyond."""
    g = torch.Generator(device=gpu).manual_seed(m * n + k)
    qw = torch.randint(-(2**31), 2**31, (n // 4, k // 8, 4), dtype=torch.int32, device=gpu, generator=g)
    qs = torch.rand(k // 128, n // 4, 4, device=gpu, generator=g) * 0.01 + 0.001
    qz = torch.randint(0, 16, (k // 128, n // 4, 4), dtype=torch.int8, device=gpu, generator=g)
    x = torch.randn(m, k, device=gpu, generator=g).to(dtype)
    y = fused_ops.int4_gemv_tiled(x, qw, qs, qz, 128, k, n)
    codes = torch.stack([(qw >> (4 * j)) & 15 for j in range(8)], dim=2).permute(0, 3, 1, 2).reshape(n, k)
    zeros, scales = (t.reshape(k // 128, n).t().repeat_interleave(128, dim=1).double() for t in (qz, qs))
    ref = x.double() @ ((codes - zeros) * scales).t()
    # half a unit of the result's last place, and fp32 sums of x (128 + code) and x (128 + zero), no more than
    # 128 roundings one after the other in either
    bound = ref.abs() * (2.0**-8 if dtype == torch.bfloat16 else 2.0**-11) + \
        (x.double().abs() @ scales.t()) * 2 * 143 * 128 * 2.0**-24
    assert bool(((y.double() - ref).abs() <= bound).all())
