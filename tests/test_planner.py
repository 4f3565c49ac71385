"""The decode planner's choices (host code, no GPU): how a small batch is split
and when an uneven one goes page-balanced."""
import ctypes

import pytest

from gllm_amd import _lib

CUS = 256      # what the planner assumes without a device


def _info(q, L, Hq=32, Hkv=8, D=128, split=0, hw=0):
    lib = _lib.load()
    h = ctypes.c_void_p()
    arr = lambda v: (ctypes.c_int32 * len(v))(*v)
    _lib.check(lib.gllm_attn_plan_create(ctypes.byref(h), arr(q), arr(L), len(L), 0, Hq, Hkv, D, 16,
                                         _lib.DTYPE_BF16, split, hw))
    out = (ctypes.c_int64 * 10)()
    _lib.check(lib.gllm_attn_plan_info(h, out, 10))
    nbytes = lib.gllm_attn_plan_workspace_bytes(h)
    lib.gllm_attn_plan_destroy(h)
    keys = ("items", "split", "dec", "pre", "partials", "rows", "hw", "dw", "pw", "segs")
    return dict(zip(keys, out)), nbytes


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("L", [[1], [127], [300], [2048], [40000], [5000, 3000, 7000, 4200], [500] * 16, [3000] * 16])
def test_small_batches_get_one_item_per_cu(L, D):
    i, nbytes = _info([1] * len(L), L, D=D)
    assert i["segs"] == 0 and i["dec"] == len(L)
    assert i["items"] <= CUS
    if i["partials"] == 0:               # a split would shed less than 128 KB of K/V from the longest item
        assert i["items"] == len(L) * -(-8 // i["hw"])
        return
    # splits of at least 128 keys, and no coarser than the CUs ask for
    assert i["split"] >= 128
    if i["split"] > 128:
        finer = sum(-(-x // (i["split"] - 32)) for x in L) * -(-8 // i["hw"])
        assert finer > CUS
    assert nbytes >= i["partials"] * 16 * (D + 2) * 4


@pytest.mark.parametrize("D,last_whole,first_split", [(64, 320, 448), (128, 192, 320)])
@pytest.mark.parametrize("B", [1, 8, 16])
def test_short_sequences_stay_whole(B, D, last_whole, first_split):
    assert _info([1] * B, [last_whole] * B, D=D)[0]["partials"] == 0
    assert _info([1] * B, [first_split] * B, D=D)[0]["partials"] > 0


def test_uneven_batches_go_page_balanced():
    import random
    r = random.Random(0)
    uneven = [r.randint(500, 3000) for _ in range(32)]
    assert _info([1] * 32, uneven)[0]["segs"] > 0
    assert _info([1] * 32, [1500] * 32)[0]["segs"] == 0          # one equal item per CU
    assert _info([1] * 40, [4000] * 40)[0]["segs"] > 0           # 1.25 rounds of long items
    assert _info([1] * 32, uneven, split=1024)[0]["segs"] == 0   # a split length was asked for
    assert _info([1] * 31 + [64], uneven)[0]["segs"] == 0        # mixed batches only on request
    # ... but a mixed batch whose decodes leave CUs far behind is split
    skew = [r.randint(300, 600) for _ in range(56)] + [8000] * 8
    assert _info([1] * 64 + [256], skew + [2000])[0]["split"] < 8000
    assert _info([1] * 64 + [256], [600] * 64 + [2000])[0]["split"] > 600
    many = [r.randint(256, 4096) for _ in range(256)]
    assert _info([1] * 256, many)[0]["segs"] == 0                # four items per CU even out


@pytest.mark.parametrize("hidden,heads", [(4096, 32), (3072, 24), (5120, 40), (8192, 64), (2048, 16), (1024, 8)])
def test_qkv_split_fits_the_noalloc_scratch(hidden, heads):
    """A batch whose partials fit 24 MiB at about two workgroups per CU fits
    them at the count that is chosen."""
    lib = _lib.load()
    for n in list(range(33, 700, 7)) + [256, 320, 512]:
        F = (heads + 16) * 128
        wgs = -(-n // 64) * (heads + 16)
        want = min(-(-2 * CUS // wgs), hidden // 256, 16)
        got = lib.gllm_qkv_workspace_bytes(n, hidden, heads, 8, 128, 1)
        assert got % (n * F * 4) == 0 and got // (n * F * 4) <= 16
        if want * n * F * 4 <= 24 << 20:
            assert got <= 24 << 20, (n, got)


@pytest.mark.parametrize("Hq,Hkv,D,behind,ahead", [
    (32, 8, 128, [3984, 4096, 12286, 12288, 13627, 15718, 15884, 16384], [4100, 5282, 8200, 10362, 16390, 17099, 19679]),
    (24, 8, 128, [15748, 16384], [3072, 3148, 3244, 5377, 6043, 16390, 18608]),
    (32, 8, 64, [], [3072, 4096, 5186, 5377, 9768, 16384, 19352]),
    (32, 2, 128, [3798, 4096, 7397, 16384], [3148, 4100, 8436, 9003, 19352]),
    (4, 4, 64, [], [3072, 8192, 19679]), (2, 2, 128, [], [3072, 6000, 19679])])
def test_prompt_projections_where_the_library_is_ahead(Hq, Hkv, D, behind, ahead):
    """Token counts measured on either side: the tiles' rounds nearly empty, or
    the library's full, and the other way round."""
    lib = _lib.load()
    assert [n for n in behind if lib.gllm_qkv_tiles_ahead(n, Hq, Hkv, D)] == []
    assert [n for n in ahead if not lib.gllm_qkv_tiles_ahead(n, Hq, Hkv, D)] == []
    assert lib.gllm_qkv_tiles_ahead(0, Hq, Hkv, D) == 0 and lib.gllm_qkv_tiles_ahead(4096, Hq, 0, D) == 0
    assert lib.gllm_qkv_tiles_ahead(4096, Hq, Hkv, 96) == 0
