"""The generic attention kernels at the edges of their tiles and of the choice
between them: 16 (query row, head) columns per stream workgroup, 128 per tiled
one, 16- and 32-key steps, the padded head dims, vector and element loads, and
both sides of the tiled kernel's workgroup count."""
import pytest
import torch

import gllm_amd
from gllm_amd import paged
from oracle import attention as oa
from tests.gpu_helpers import assert_close_bf16, make_batch, oracle_paged

pytestmark = pytest.mark.gpu
DEV = "cuda"
F32, BF, F16 = torch.float32, torch.bfloat16, torch.float16

FEW = ([0, 15, 16, 17, 31, 200], [1, 2, 17, 33, 16, 1])            # stream kernel only
MANY = ([0, 3, 64, 31, 250, 7], [300, 17, 16, 257, 129, 1])        # tiled sequences and stream ones


def _check(out, ref, what):
    # fp32 both sides: weights carry a few ulps (scores below ~8), sums over at
    # most ~400 keys of values below ~5: well under 1e-4
    if out.dtype == F32:
        assert (out.cpu() - ref).abs().max().item() < 1e-4, what
    else:
        assert_close_bf16(out, ref, what)


@pytest.mark.parametrize("ctx,ql", [FEW, MANY])
@pytest.mark.parametrize("dtype,kv,D,Hq,Hkv", [
    (F32, F32, 64, 32, 8), (F32, F32, 128, 12, 12), (F32, F32, 50, 16, 8), (F32, BF, 96, 32, 8), (F32, F32, 256, 16, 4),
    (BF, BF, 80, 32, 8), (BF, BF, 256, 32, 8), (F16, F16, 96, 40, 8), (BF, F32, 64, 32, 8), (F16, BF, 128, 32, 8),
    (BF, torch.float8_e4m3fn, 32, 32, 8), (F16, F16, 6, 64, 2)])
def test_paged(ctx, ql, dtype, kv, D, Hq, Hkv):
    b = make_batch(ctx, ql, Hq, Hkv, D, dtype=dtype)
    if kv != dtype:
        b.k_cache, b.v_cache = b.k_cache.to(kv), b.v_cache.to(kv)
    plan = paged.AttentionPlan(b.q_lens, b.seq_lens, num_q_heads=Hq, num_kv_heads=Hkv, head_dim=D, block_size=16,
                               dtype=dtype, device=DEV)
    out = paged.paged_attention(plan, b.q, b.k_cache, b.v_cache, b.block_table)
    b.k_cache, b.v_cache = b.k_cache.to(dtype), b.v_cache.to(dtype)     # the gather's cast
    _check(out, oracle_paged(b), f"{dtype} {kv} {D}")


@pytest.mark.parametrize("ctx,ql", [([0, 63, 300, 17, 4], [32, 1, 1, 1, 2]),    # 8 column groups at G = 4, odd with one more
                                    ([5, 0, 40], [1, 45, 1]), ([8, 130, 65], [16, 1, 3])])
@pytest.mark.parametrize("dtype,D", [(F32, 64), (BF, 80)])
def test_decodes_beside_a_chunk(ctx, ql, dtype, D):
    test_paged(ctx, ql, dtype, dtype, D, 32, 8)


def test_paged_unaligned_rows():
    """Cache rows at odd element offsets: the element loads of both kernels."""
    for ctx, ql in (FEW, MANY):
        b = make_batch(ctx, ql, 32, 8, 64, dtype=F32)
        ns = b.k_cache.shape[0]
        wide = torch.zeros(2, ns, 8 * 64 + 1, device=DEV)
        caches = []
        for w, c in zip(wide, (b.k_cache, b.v_cache)):
            view = w[:, 1:].unflatten(1, (8, 64))
            view.copy_(c)
            caches.append(view)
        plan = paged.AttentionPlan(b.q_lens, b.seq_lens, num_q_heads=32, num_kv_heads=8, head_dim=64, block_size=16,
                                   dtype=F32, device=DEV)
        out = paged.paged_attention(plan, b.q, caches[0], caches[1], b.block_table)
        _check(out, oracle_paged(b), "unaligned")


@pytest.mark.parametrize("dtype,kv,D,off", [
    (F32, F32, 2, 0), (BF, BF, 2, 1), (BF, BF, 50, 0), (BF, torch.float8_e4m3fn, 34, 3), (F16, F16, 126, 0),
    (BF, BF, 130, 1), (F16, F32, 250, 0), (F32, F32, 254, 1), (F16, F16, 96, 1), (BF, F32, 64, 1)])
def test_paged_odd_head_dims_and_rows(dtype, kv, D, off):
    """Head dims that are no multiple of 4 and rows at odd offsets: the last row
    of the pool ends where its buffer does, so a load past a row's end would be
    past the buffer's."""
    for ctx, ql in (FEW, MANY):
        b = make_batch(ctx, ql, 16, 4, D, dtype=dtype)
        ns, row = b.k_cache.shape[0], 4 * D
        caches = []
        for c in (b.k_cache, b.v_cache):
            buf = torch.zeros(ns * (row + off) + off, device=DEV).to(kv)
            view = buf[off:].unflatten(0, (ns, row + off))[:, :row].unflatten(1, (4, D))
            view.copy_(c.to(kv))
            caches.append(view)
        plan = paged.AttentionPlan(b.q_lens, b.seq_lens, num_q_heads=16, num_kv_heads=4, head_dim=D, block_size=16,
                                   dtype=dtype, device=DEV)
        out = paged.paged_attention(plan, b.q, caches[0], caches[1], b.block_table)
        b.k_cache, b.v_cache = (c.contiguous().to(dtype) for c in caches)
        _check(out, oracle_paged(b), f"{dtype} {kv} {D} +{off}")


@pytest.mark.parametrize("dtype", [F32, BF])
@pytest.mark.parametrize("B,Tq,T,Hq,Hkv,D", [(1, 5, 33, 8, 2, 48), (2, 40, 65, 8, 2, 80), (3, 300, 333, 32, 8, 96)])
def test_dense_masks(dtype, B, Tq, T, Hq, Hkv, D):
    """Dense bias with masked keys, a fully masked row (NaN) and a row of the
    type's lowest value (uniform weights), on both kernels."""
    g = torch.Generator().manual_seed(T)
    q, k, v = (torch.randn(B, n, h, D, generator=g).to(dtype) for n, h in ((Tq, Hq), (T, Hkv), (T, Hkv)))
    bias = torch.where(torch.rand(B, Tq, T, generator=g) < 0.3, float("-inf"), 0.25).to(dtype)
    bias[..., 0] = 0.0
    bias[0, 1] = float("-inf")
    bias[0, 2] = torch.finfo(dtype).min
    ref = oa.reference_attention(q.float(), k.float(), v.float(), bias.float())
    out = gllm_amd.reference_attention(q.to(DEV), k.to(DEV), v.to(DEV), bias.to(DEV)).cpu()
    assert torch.isnan(out[0, 1]).all() and torch.isnan(ref[0, 1]).all()
    fin = torch.isfinite(ref)
    _check(out[fin], ref[fin], f"dense {dtype}")
