"""Which kernel a Python call reaches and with what strides (no GPU: a recorder
stands in for the library)."""
import pytest
import torch

from gllm_amd import _lib, paged

BF = torch.bfloat16


class Recorder:
    """Every entry point succeeds and is noted with its arguments."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            self.calls.append((name, args))
            return 0
        return call

    def names(self):
        return [n for n, _ in self.calls if n != "gllm_qkv_workspace_bytes"]


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
