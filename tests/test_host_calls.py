"""Which kernel a Python call reaches and with what strides (no GPU: a recorder
stands in for the library)."""
import pytest
import torch

import gllm_amd
from gllm_amd import _lib, paged

BF = torch.bfloat16


class Recorder:
    """Every entry point succeeds and is noted with its arguments."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            self.calls.append((name, args))
            return int(name == "gllm_qkv_tiles_ahead")
        return call

    def names(self):
        return [n for n, _ in self.calls if n not in ("gllm_qkv_workspace_bytes", "gllm_qkv_tiles_ahead")]


@pytest.fixture
def lib(monkeypatch):
    rec = Recorder()
    monkeypatch.setattr(_lib, "load", lambda: rec)
    monkeypatch.setattr(_lib, "stream_ptr", lambda dev: 0)
    return rec


def _caches(slots, Hkv, D, dtype=BF):
    return torch.zeros(slots, Hkv, D, dtype=dtype), torch.zeros(slots, Hkv, D, dtype=dtype)


def test_one_row_of_a_wider_table(lib):
    """One cos / sin row, or one token row, cut out of wider rows is a whole row:
    its stride means nothing."""
    kc, vc = _caches(32, 4, 64)
    wide, own = torch.zeros(9, 64, dtype=BF), torch.zeros(1, 32, dtype=BF)
    cos, slots = wide[5:6, :32], torch.zeros(1, dtype=torch.int64)
    assert cos.stride(0) != own.stride(0)
    k = torch.zeros(1, 4, 64, dtype=BF)
    paged.rope_kv_write(k, k, cos, own, kc, vc, slots)
    paged.rope_rotate(k, cos, own)
    x = torch.zeros(3, 260, dtype=BF)[:1, :256]          # rows 260 elements apart: no multiple of 8
    w = torch.zeros(256, 256, dtype=BF)
    paged.qkv_rope_kv_write(x, w, w, w, cos, own, kc, vc, slots)
    name, args = lib.calls[-1]
    assert name == "gllm_qkv_rope_kv_write" and args[1] == 256


def _qkv(lib, n=paged.QKV_UNFUSED_FROM, x=None, **kw):
    """A projection call that the large tiles take; the entry points it reached."""
    hidden, H, D = 64, 4, 64
    x = torch.zeros(n, hidden, dtype=BF) if x is None else x
    w = torch.zeros(H * D, hidden, dtype=BF)
    kc, vc = _caches(16, H, D)
    tab, slots = torch.zeros(n, D // 2, dtype=BF), torch.zeros(n, dtype=torch.int64)
    paged.qkv_rope_kv_write(x, w, w, w, tab, tab, kc, vc, slots, **kw)
    return lib.names()


def test_projection_of_expanded_rows(lib):
    """Token rows that overlap (a row expanded) are the library's at prompt sizes:
    the kernels refuse row strides below the hidden size."""
    row = torch.zeros(1, 64, dtype=BF)
    n = paged.QKV_UNFUSED_FROM
    assert _qkv(lib) == ["gllm_qkv_rope_kv_write"]
    lib.calls.clear()
    assert _qkv(lib, x=row.expand(n, 64)) == ["gllm_rope_kv_write"]


def test_explicit_threshold_forces_the_library(lib):
    """A threshold the caller gives holds as it stands; only the default lets the
    large tiles take prompts beyond it."""
    n = paged.QKV_UNFUSED_FROM
    for given in (n, int("3072"), 100, 1):
        lib.calls.clear()
        assert _qkv(lib, unfused_from=given) == ["gllm_rope_kv_write"], given
    for kw in ({}, {"unfused_from": None}, {"unfused_from": n + 1}):
        lib.calls.clear()
        assert _qkv(lib, **kw) == ["gllm_qkv_rope_kv_write"], kw


class _Plan:
    """What a layer asks of the step's plan (kept on the metadata)."""
    block_size, dtype, max_query_len = 16, BF, 1

    def __init__(self, Hq, Hkv, D):
        self.num_q_heads, self.num_kv_heads, self.head_dim = Hq, Hkv, D


def _forward(monkeypatch, cls=gllm_amd.Attention, rows=2, Hq=4, Hkv=2, D=64, dev="meta", slots_dev="meta", ql_dev="meta",
             patch=None, pool=None):
    """The calls one decode step of a layer makes, tensors without storage."""
    calls = []

    def note(name, out):
        def call(*args, **kw):
            calls.append(name + ("+kv" if kw.get("kv_new") is not None else ""))
            return out
        return call

    class Cfg:
        num_attn_heads, num_kv_heads, head_dim, hidden_size, dtype = Hq, Hkv, D, Hq * D, BF

    hid = Hq * D
    w = {f"model.layers.0.self_attn.{n}_proj.weight": torch.zeros(h * D, hid, dtype=BF, device=dev)
         for n, h in (("q", Hq), ("k", Hkv), ("v", Hkv), ("o", Hq))}
    att = cls(0, Cfg, w)
    out = torch.zeros(rows, 1, Hq, D, dtype=BF, device=dev)
    monkeypatch.setattr(paged, "qkv_rope_kv_write", note("fused projection", out))
    monkeypatch.setattr(paged, "paged_attention", note("attention", out))
    if patch:
        patch(att, note("override", out))
    meta = gllm_amd.AttentionMetadata(
        query_lens=torch.ones(rows, dtype=torch.int32, device=ql_dev), seq_lens=torch.ones(rows, dtype=torch.int32),
        max_seq_len=1, block_table=torch.zeros(rows, 1, dtype=torch.int32, device=dev), slot_mapping=None,
        query_slot_mapping=torch.zeros(rows, 1, dtype=torch.int64, device=slots_dev), bias=None, block_size=16)
    meta._gllm_plan = _Plan(Hq, Hkv, D)
    tab = torch.zeros(rows, 1, D // 2, dtype=BF, device=dev)
    att.forward(torch.zeros(rows, 1, hid, dtype=BF, device=dev), tab, tab,
                torch.zeros(2, 32, Hkv, D, dtype=BF, device=dev) if pool is None else pool, meta)
    return calls


def test_forward_reads_no_host_metadata(monkeypatch):
    """Slots and query lengths on the host stay with the route that takes the
    slots from the block table: the fused projection reads both on the GPU."""
    assert _forward(monkeypatch) == ["fused projection", "attention"]
    assert _forward(monkeypatch, slots_dev="cpu") == ["attention+kv"]
    assert _forward(monkeypatch, ql_dev="cpu") == ["attention+kv"]


def test_forward_reaches_an_overridden_attention(monkeypatch):
    """A subclass's, or one object's, own ``attention`` is called on every step."""
    class Own(gllm_amd.Attention):
        def attention(self, *args):
            self.seen = True
            return super().attention(*args)

    seen = []
    assert _forward(monkeypatch, cls=Own, patch=lambda att, call: seen.append(att)) == ["attention+kv"]
    assert seen[0].seen
    assert _forward(monkeypatch, patch=lambda att, call: setattr(att, "attention", call)) == ["override"]


def test_forward_takes_caches_of_unlike_length(monkeypatch):
    """K and V pools given as a pair may differ in their number of slots."""
    pool = tuple(torch.zeros(n, 2, 64, dtype=BF, device="meta") for n in (32, 48))
    assert _forward(monkeypatch, pool=pool) == ["attention+kv"]


def test_forward_projects_with_the_library_where_it_is_ahead(monkeypatch):
    """Wide layers: the fused kernels for up to 256 rows, F.linear beyond."""
    fused, linear = ["fused projection", "attention"], ["attention+kv"]
    wide, wider = dict(Hq=64, Hkv=8, D=128), dict(Hq=64, Hkv=64, D=128)
    assert _forward(monkeypatch, rows=256, **wide) == fused
    for rows in (257, 512, 3000):
        assert _forward(monkeypatch, rows=rows, **wide) == linear
    assert _forward(monkeypatch, rows=1, **wider) == linear
    for Hq in (16, 32):
        assert _forward(monkeypatch, rows=3000, Hq=Hq, Hkv=8, D=128) == fused
    assert _forward(monkeypatch, rows=paged.QKV_UNFUSED_FROM) == linear
