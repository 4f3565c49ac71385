"""bf16 prefill at head dim 64 on either side of the line from which two
workgroups share a CU (512 items of at most 320 keys on average on 256 CUs, or
2,048 items without cached context): many short prompts, ragged ends, cached
context, scores far outside the softmax's fast range."""
import pytest
import torch

from gllm_amd import paged
from gpu_helpers import assert_close_bf16, make_batch, oracle_paged

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Hq,Hkv,ctx,ql,grow", [
    (32, 8, [0] * 64, [64] * 63 + [33], 1.0), (32, 8, [0] * 63, [64] * 63, 1.0),        # 512 items, 504
    (32, 8, [0, 37] * 33, [64, 20] * 33, 30.0), (8, 8, [0] * 70, [17, 100] * 35, 1.0),
    (32, 8, [800] * 64, [64] * 64, 1.0), (64, 8, [0] * 6, [1400] * 6, 1.0)])
def test_short_prompts(Hq, Hkv, ctx, ql, grow):
    print(f"prefill pairs {Hq}/{Hkv} {len(ql)} x {ql[0]} on {ctx[0]}", flush=True)
    b = make_batch(ctx, ql, Hq, Hkv, 64)
    b.q.mul_(grow)
    plan = paged.AttentionPlan(b.q_lens, b.seq_lens, num_q_heads=Hq, num_kv_heads=Hkv, head_dim=64,
                               block_size=16, dtype=torch.bfloat16, device="cuda")
    out = paged.paged_attention(plan, b.q, b.k_cache, b.v_cache, b.block_table)
    torch.cuda.synchronize()
    assert_close_bf16(out, oracle_paged(b), "prefill")
