"""Split partials: one to many per (sequence, head), merged by one group of
threads (up to 8 splits) or several, for the fewest and the most query rows of
the decode path, under split and page-balanced plans."""
import pytest
import torch

from gllm_amd import paged
from tests.gpu_helpers import assert_close_bf16, make_batch, oracle_paged

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Hq,Hkv,ql", [(32, 8, [1, 4, 2]), (12, 12, [16, 1, 9]), (16, 1, [1, 1, 1]), (20, 5, [4, 1, 1])])
@pytest.mark.parametrize("split,hw", [(32, 1), (64, 2), (256, 4), (paged.BALANCED, 0), (paged.BALANCED, 2)])
def test_merge(D, Hq, Hkv, ql, split, hw):
    b = make_batch([1500, 40, 290], ql, Hq, Hkv, D)     # up to 47, 2 and 10 splits of 32
    plan = paged.AttentionPlan(b.q_lens, b.seq_lens, num_q_heads=Hq, num_kv_heads=Hkv, head_dim=D, block_size=16,
                               dtype=torch.bfloat16, device=DEV, split_tokens=split, heads_per_wg=hw)
    assert plan.info["partials"] > 0
    for _ in range(2):
        out = paged.paged_attention(plan, b.q, b.k_cache, b.v_cache, b.block_table)
        assert_close_bf16(out, oracle_paged(b), f"{split} {hw}")
