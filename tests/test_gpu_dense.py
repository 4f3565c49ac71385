"""The dense-bias op on the MFMA kernels at the edges of its column groups (32
(row, head) pairs per wave, 256 per workgroup) and key tiles, with bias rows
that 8-byte loads may read and ones they may not."""
import pytest
import torch

import gllm_amd
from oracle import attention as oa
from tests.gpu_helpers import assert_close_bf16

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("Tq,T,Hq,Hkv,D", [(1, 4, 32, 8, 64), (7, 65, 6, 2, 128), (33, 128, 32, 8, 64),
                                           (64, 131, 5, 5, 64), (65, 196, 40, 8, 128)])
def test_dense_edges(dtype, off, Tq, T, Hq, Hkv, D):
    g = torch.Generator().manual_seed(Tq + T)
    q, k, v = (torch.randn(2, n, h, D, generator=g).to(dtype) for n, h in ((Tq, Hq), (T, Hkv), (T, Hkv)))
    wide = torch.randn(2, Tq, T + 4, generator=g)
    wide[torch.rand(wide.shape, generator=g) < 0.2] = float("-inf")
    wide[..., off] = 0.0                                    # some key visible in every row
    wide = wide.to(dtype)
    ref = oa.reference_attention(q.float(), k.float(), v.float(), wide[..., off:off + T].float())
    out = gllm_amd.reference_attention(q.to(DEV), k.to(DEV), v.to(DEV), wide.to(DEV)[..., off:off + T])
    assert_close_bf16(out, ref, f"dense {Tq} {T} {D} offset {off}")
