"""Attention.forward on decode batches: the fused projection route (bf16) at
the edges of its kernels' token counts against the same layer through
F.linear, and the calls that keep that route."""
import pytest
import torch
import torch.nn.functional as F

import gllm_amd
from tests.gpu_helpers import assert_close_bf16

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF, F16, F8 = torch.bfloat16, torch.float16, torch.float8_e4m3fn


def _layer(B, Tq, Hq, Hkv, D, dtype, kv, odd=False):
    g = torch.Generator().manual_seed(B)
    hid, bs = Hq * D, 16
    L = [int(x) + Tq for x in torch.randint(0, 200, (B,), generator=g)]
    need = [-(-x // bs) for x in L]
    perm = torch.randperm(sum(need), generator=g).int() + 1
    bt = torch.zeros(B, max(need), dtype=torch.int32)
    o = 0
    for i, n in enumerate(need):
        bt[i, :n] = perm[o:o + n]
        o += n
    pos = torch.tensor([[x - Tq + r for r in range(Tq)] for x in L])
    slots = torch.gather(bt.long(), 1, pos // bs) * bs + pos % bs

    class Cfg:
        num_attn_heads, num_kv_heads, head_dim, hidden_size = Hq, Hkv, D, hid

    Cfg.dtype = dtype
    w = {}
    for n, rows in (("q", hid), ("k", Hkv * D), ("v", Hkv * D), ("o", hid)):
        t = (torch.randn(rows, hid, generator=g) / hid ** 0.5).to(dtype).to(DEV)
        if odd:                     # a weight whose rows start 2 bytes off
            t = F.pad(t, (1, 7))[:, 1:1 + hid]
        w[f"model.layers.0.self_attn.{n}_proj.weight"] = t
    meta = gllm_amd.AttentionMetadata(torch.full((B,), Tq, dtype=torch.int32, device=DEV),
                                      torch.tensor(L, dtype=torch.int32, device=DEV), max(L), bt.to(DEV), None,
                                      slots.to(DEV), None, bs)
    ang = pos.unsqueeze(-1) * 500000.0 ** (-2 * torch.arange(D // 2) / D)
    pool = torch.randn(2, (sum(need) + 1) * bs, Hkv, D, generator=g).to(dtype).to(kv).to(DEV)
    x = torch.randn(B, Tq, hid, generator=g).to(dtype).to(DEV)
    return gllm_amd.Attention(0, Cfg, w), x, ang.cos().to(dtype).to(DEV), ang.sin().to(dtype).to(DEV), pool, meta


def _routes(att):
    """What each call of forward's fused route returned."""
    seen, fused = [], att._fused_decode

    def spy(*args):
        seen.append(fused(*args))
        return seen[-1]
    att._fused_decode = spy
    return seen


def _by_linear(att, x, cos, sin, pool, meta):
    B, Tq, _ = x.shape
    q, k, v = (F.linear(x, w).view(B, Tq, -1, att.head_dim) for w in (att.W_q, att.W_k, att.W_v))
    return F.linear(att.attention(q, k, v, cos, sin, pool, meta).view(B, Tq, -1), att.W_o)


@pytest.mark.parametrize("B,Tq", [(1, 1), (32, 1), (33, 1), (65, 1), (5, 4)])
@pytest.mark.parametrize("Hq,Hkv,D,kv", [(16, 4, 64, BF), (8, 2, 128, BF), (8, 2, 128, F8)])
def test_fused_decode(B, Tq, Hq, Hkv, D, kv):
    att, x, cos, sin, pool, meta = _layer(B, Tq, Hq, Hkv, D, BF, kv)
    p1, p2 = pool.clone(), pool.clone()
    seen = _routes(att)
    out, ref = att.forward(x, cos, sin, p1, meta), _by_linear(att, x, cos, sin, p2, meta)
    assert len(seen) == 1 and seen[0] is not None
    assert_close_bf16(out, ref, "forward")
    # the written rows: projections summed in another order, so a step of the
    # cache dtype on few values (bf16 2^-7 after the rotation's roundings, fp8 2^-3)
    d = (p1.float() - p2.float()).abs()
    step = 2.0 ** (-3 if kv == F8 else -6)
    assert (d <= step * torch.maximum(p1.float().abs(), p2.float().abs()).clamp(min=0.25)).all()
    assert (d > 0).float().mean() < 0.02


@pytest.mark.parametrize("dtype,odd", [(F16, False), (BF, True)])
def test_other_calls_keep_their_route(dtype, odd):
    att, x, cos, sin, pool, meta = _layer(9, 1, 8, 2, 64, dtype, dtype, odd)
    p1, p2 = pool.clone(), pool.clone()
    seen = _routes(att)
    assert torch.equal(att.forward(x, cos, sin, p1, meta), _by_linear(att, x, cos, sin, p2, meta))
    assert torch.equal(p1, p2)
    assert seen in ([], [None])
