"""Generic attention of 16-bit models where the last bits of the probabilities
decide the result."""
import math

import pytest
import torch

import gllm_amd
from gllm_amd import paged

pytestmark = pytest.mark.gpu
DEV = "cuda"
F32, BF, F16 = torch.float32, torch.bfloat16, torch.float16
BS = 16


def run(q, k, v, dtype, kv=None, kv_new=None):
    """Every row of q [rows, Hq, D] over the keys k / v [n, Hkv, D] (the rows are
    the last ones), in scattered blocks."""
    n, Hkv, D = k.shape
    rows, Hq = q.shape[:2]
    nb = -(-n // BS)
    table = torch.randperm(nb, generator=torch.Generator().manual_seed(n)).int() + 1
    slot = table.long()[torch.arange(n) // BS] * BS + torch.arange(n) % BS
    caches = []
    for t in (k, v):
        c = torch.zeros((nb + 1) * BS, Hkv, D, dtype=kv or dtype)
        c[slot] = t.to(kv or dtype)
        caches.append(c.to(DEV))
    plan = paged.AttentionPlan([rows], [n], num_q_heads=Hq, num_kv_heads=Hkv, head_dim=D, block_size=BS, dtype=dtype,
                               device=DEV)
    new = None if kv_new is None else tuple(t.to(dtype).to(DEV) for t in kv_new)
    return paged.paged_attention(plan, q.to(dtype).to(DEV), *caches, table.view(1, -1).to(DEV), kv_new=new).cpu()


@pytest.mark.parametrize("D", [96, 256])
@pytest.mark.parametrize("shift", [10, 17, 21, 23])
def test_f16_small_weights(shift, D):
    """One key takes almost all of the weight and has V = 0: the result is the
    sum of 1,500 equal weights just above 2^-shift, an fp16 subnormal from shift
    15 on.  fp32 weights: only the output's rounding is left."""
    n, Hq = 1501, 4
    g = torch.Generator().manual_seed(shift)
    k = torch.zeros(n, 1, D)
    q = torch.zeros(1, Hq, D)
    q[..., 0] = torch.tensor([(shift - h / 5) * math.log(2) for h in range(Hq)]).half().float()
    k[700, 0, 0] = math.sqrt(D)                      # score q[0] there, 0 elsewhere
    k = k.half().float()
    v = 1.0 + torch.rand(n, 1, D, generator=g).half().float()
    v[700] = 0.0
    out = run(q, k, v, F16).double()
    s = (q[0].double() @ k[:, 0].double().t()) / math.sqrt(D)
    ref = torch.softmax(s, -1) @ v[:, 0].half().double()
    # one fp16 rounding, 2^-11 of the value (or half a subnormal step), and a few fp32 ulps of the weights
    assert ((out[0] - ref).abs() <= ref.abs() * 2.0 ** -10.9 + 2.0 ** -24).all(), ((out[0] - ref) / ref).abs().max()


@pytest.mark.parametrize("D,kv", [(96, BF), (256, BF), (128, F32)])
def test_bf16_differences_of_weights(D, kv):
    """Keys in pairs whose weights differ by 2^-13 / sqrt(D) of themselves and
    whose V cancel but for that: the weights' last bits are the result."""
    n, Hq = 128, 32
    g = torch.Generator().manual_seed(D)
    k = torch.randn(n // 2, 1, D, generator=g).to(BF).float().repeat_interleave(2, 0)
    k[0::2, 0, 0], k[1::2, 0, 0] = 0.0, 1.0
    q = torch.randn(1, Hq, D, generator=g).to(BF).float()
    q[..., 0] = 2.0 ** -13
    v = torch.ones(n, 1, D)
    v[0::2] = -1.0
    out = run(q, k, v, BF, kv)[0, :, 0].double()
    s = (q[0].double() @ k[:, 0].double().t()) / math.sqrt(D)
    ref = torch.softmax(s, -1) @ v[:, 0, 0].double()
    rel = (out - ref) / ref
    # bf16's rounding is at most 2^-9 of the result; an fp32 ulp of a score or a
    # weight is up to ~2^-6 of a pair's difference, in either direction over 64 pairs
    assert rel.square().mean().sqrt() < 0.01, rel


@pytest.mark.parametrize("dtype,kv,D", [(BF, BF, 96), (BF, F32, 64), (F16, F16, 256), (F32, F32, 64), (BF, BF, 50)])
@pytest.mark.parametrize("rows,n,fused", [(1, 64, False), (3, 80, False), (200, 256, False),
                                          (1, 37, True), (3, 50, True), (16, 64, True)])
def test_infinities_in_v(dtype, kv, D, rows, n, fused):
    """An infinity in V at a key that every row sees is the result in its dim, as
    weight times infinity is for any weight above 0: at the first key, at the one
    that takes the largest weight and at the last row's own key, also where that is
    the new token which the launch writes, whatever the number of keys."""
    g = torch.Generator().manual_seed(n)
    Hq, Hkv = 64, 16                                 # tiled from ~190 rows on
    q = torch.randn(rows, Hq, D, generator=g)
    k, v = torch.randn(n, Hkv, D, generator=g), torch.randn(n, Hkv, D, generator=g)
    top = n - rows                                   # the newest key that every row sees
    k[5] *= 4.0 / math.sqrt(D)
    k[5, :, 0] += 3.0
    q[..., 0] += 3.0
    v[0, :, 1], v[5, :, 2], v[top, :, 3], v[n - 1, :, 4] = math.inf, -math.inf, math.inf, -math.inf
    q, k, v = (t.to(dtype) for t in (q, k, v))
    if not fused:
        out = run(q, k, v, dtype, kv)
    else:                                            # the new rows' keys come with the call
        kc, vc = k.clone(), v.clone()
        kc[n - rows:], vc[n - rows:] = 0.0, 0.0
        out = run(q, kc, vc, dtype, kv, kv_new=(k[n - rows:], v[n - rows:]))
    assert (out[..., 1] == math.inf).all() and (out[..., 2] == -math.inf).all() and (out[..., 3] == math.inf).all()
    assert (out[-1, :, 4] == -math.inf).all()        # the earlier rows give it weight 0: NaN, as in the reference
    assert torch.isfinite(out[..., 5:].float()).all() and torch.isfinite(out[..., 0].float()).all()


@pytest.mark.parametrize("B,Tq,D,part", [(1, 1, 64, 2), (1, 1, 128, 4), (1, 1, 256, 4), (3, 300, 256, 4)])
def test_f32_score_sums_are_short(B, Tq, D, part):
    """Key 0's score is 256 plus D - 4 products of 2^-17, each lost when it is added
    to the 256 (half an ulp is 2^-16); key 1's is the exact sum.  The result, (p0 - p1)
    / (p0 + p1), shows how many met the 256: the dims of one partial sum, D / part."""
    n = D - 4
    q, k = torch.zeros(B, Tq, 32, D), torch.zeros(B, 2, 8, D)
    q[..., 0], q[..., 1:n + 1] = 16.0, 2.0 ** -8
    k[:, 0, :, 0], k[:, 0, :, 1:n + 1] = 16.0, 2.0 ** -9
    k[:, 1, :, 0] = 16.0 + n * 2.0 ** -21              # a multiple of fp32's 2^-19 there
    v = torch.ones(B, 2, 8, D)
    v[:, 1] = -1.0
    out = gllm_amd.reference_attention(q.to(DEV), k.to(DEV), v.to(DEV), torch.zeros(B, Tq, 2, device=DEV)).cpu()
    lost = out.double().abs() * 2 * math.sqrt(D) * 2.0 ** 17   # s1 - s0 = lost 2^-17 / sqrt(D); tanh(x / 2) = x / 2 here
    # an ulp of a scaled score (2^-20 at 16, 2^-19 at 32) is 2 of these at most, and
    # each of the two scores is rounded once; the weights' ulps are a tenth of that
    assert lost.max() <= D / part + 4, lost.max()
