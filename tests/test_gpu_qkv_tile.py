"""The 256 x 256 projection tiles: small-integer data makes every dot product
exact, so q, the rotated K and V are bit-exact against the oracle; odd token
counts, one to several K slices, both head dims, an fp8 cache, padded rows."""
import pytest
import torch

from gllm_amd import paged
from oracle import rope as orope

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF, F8 = torch.bfloat16, torch.float8_e4m3fn


def _bits(t):
    return t.cpu().contiguous().view(torch.uint8 if t.element_size() == 1 else torch.int16)


@pytest.mark.parametrize("n,hidden,Hq,Hkv,D,kv,rot,pad", [
    (5633, 64, 32, 8, 128, BF, True, False), (5633, 128, 32, 8, 128, F8, False, False),
    (11000, 192, 32, 8, 64, BF, True, False), (8192, 64, 64, 8, 128, BF, True, True),
    (11000, 320, 32, 8, 64, F8, True, False)])
def test_tile256_bit_exact(n, hidden, Hq, Hkv, D, kv, rot, pad):
    g = torch.Generator().manual_seed(n + hidden)
    x = torch.randint(-1, 2, (n, hidden), generator=g).to(BF)
    w = [torch.randint(-1, 2, (h * D, hidden), generator=g).to(BF) for h in (Hq, Hkv, Hkv)]
    cos, sin = orope.rope_cache(512, D, 500000.0, BF)
    pos = torch.randint(0, 512, (n,), generator=g)
    ns = n + 40
    slots = torch.randperm(ns, generator=g)[:n]
    slots[7] = -1                                  # a slot outside the pool is not written
    real = torch.ones(n, dtype=torch.bool)
    ql = None
    if pad:                                        # [16, n / 16] rows, some of them padding
        ql = torch.randint(1, n // 16 + 1, (16,), generator=g, dtype=torch.int32)
        real = (torch.arange(n // 16)[None, :] < ql[:, None]).reshape(-1)
    kc = torch.full((ns, Hkv, D), 3.0).to(kv)
    vc = kc.clone()
    kd, vd = kc.to(DEV), vc.to(DEV)
    qd = torch.full((n, Hq, D), 9.0, dtype=BF, device=DEV)
    paged.qkv_rope_kv_write(x.to(DEV), *(t.to(DEV) for t in w), cos.to(DEV), sin.to(DEV), kd, vd, slots.to(DEV),
                            rotate_q=rot, q_out=qd, rope_rows=pos.to(DEV), unfused_from=None,
                            query_lens=None if ql is None else ql.to(DEV))
    q, k, v = ((x.float() @ t.float().t()).to(BF).view(n, -1, D) for t in w)
    rotate = lambda t: orope.apply_rope(t.unsqueeze(0), cos[pos].unsqueeze(0), sin[pos].unsqueeze(0))[0]
    q, k = rotate(q) if rot else q, rotate(k)
    ok = real & (slots >= 0)
    kc[slots[ok]], vc[slots[ok]] = k[ok].to(kv), v[ok].to(kv)
    assert torch.equal(_bits(qd)[real], _bits(q)[real]) and (qd.cpu()[~real] == 9.0).all()
    assert torch.equal(_bits(kd), _bits(kc)) and torch.equal(_bits(vd), _bits(vc))


@pytest.mark.parametrize("n,hidden,Hq,Hkv,D,kv,rot,pad", [
    (2500, 64, 40, 8, 128, BF, True, False)])   # 9 full tiles: the last round of full tiles ends short
def test_short_last_round_bit_exact(n, hidden, Hq, Hkv, D, kv, rot, pad):
    test_tile256_bit_exact(n, hidden, Hq, Hkv, D, kv, rot, pad)


@pytest.mark.parametrize("n,hidden,Hq,Hkv,D,kv,rot,pad", [
    (640, 64, 32, 8, 128, BF, True, False), (641, 64, 32, 8, 128, BF, True, False),     # one small tile per CU, over it
    (1281, 64, 32, 8, 64, F8, True, False), (1409, 64, 32, 8, 64, BF, True, False),     # two per CU at head dim 64, over it
    (768, 4096, 24, 8, 128, BF, False, False), (769, 4096, 24, 8, 128, BF, True, False),   # 0.94 and 1.1 per CU
    (1281, 4096, 24, 8, 128, F8, True, False), (1024, 5120, 24, 8, 128, BF, True, False)])   # 1.7; 1.25 of a wider layer
def test_both_sides_of_the_line_bit_exact(n, hidden, Hq, Hkv, D, kv, rot, pad):
    test_tile256_bit_exact(n, hidden, Hq, Hkv, D, kv, rot, pad)
