"""The work a serving engine has the attention path do, as measurable cases.

Every case is one call (or the few calls of one layer of one engine step)
through the package's public entry points:

- ``layer``:   ``Attention.attention`` of one decode step (padded ``[B, 1]``
               layout): RoPE, KV write and paged attention of one layer.
- ``forward``: ``Attention.forward`` of one decode step: the projections, the
               above and the output projection.
- ``paged``:   one layer's attention of a packed batch of decode sequences
               and prefill chunks: the RoPE + KV write of the new tokens and
               the paged attention (one launch for decode-only batches).
- ``qkv``:     the QKV projection fused with RoPE and the KV write.
- ``dense``:   the ``reference_attention`` op with a materialised bias.

Head shapes are those of Llama-3.2-1B (32 query / 8 KV heads of 64),
Llama-3.1-8B (32 / 8 of 128) and Llama-3.1-70B (64 / 8 of 128).  Lengths
follow from the case alone (seeded generator), values and block tables from
the seed.
"""
from __future__ import annotations

import math

import torch

import gllm_amd
from gllm_amd import paged

THETA = 500000.0
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16, "fp8": torch.float8_e4m3fn}
SIZES = {"f32": 4, "bf16": 2, "f16": 2, "fp8": 1}


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # One layer of a decode step of the fp32 1B-shaped model that the engine
        # runs for eight short chats: launch latency and host time.
        _layer("layer_decode_1b_f32", B=8, lo=20, hi=200, Hq=32, Hkv=8, D=64, dtype="f32"),
        # One whole attention layer (projections included) of an 8B model's
        # decode step for a moderately loaded server.
        _forward("forward_decode_8b", B=48, lo=128, hi=2048, Hq=32, Hkv=8, D=128, dtype="bf16"),
        # The fp32 model's prompt processing: ragged prompts, packed rows.
        _paged("prefill_1b_f32", nd=0, lo=0, hi=0, np=8, qlo=64, qhi=1024, chi=0, Hq=32, Hkv=8, D=64, dtype="f32"),
        # Interactive use: four long chats decode together.
        _paged("decode_8b_few", nd=4, lo=2048, hi=8192, np=0, qlo=0, qhi=0, chi=0, Hq=32, Hkv=8, D=128),
        # A busy 1B server's decode step.
        _paged("decode_1b", nd=64, lo=128, hi=2048, np=0, qlo=0, qhi=0, chi=0, Hq=32, Hkv=8, D=64),
        # The same over an fp8 KV cache.
        _paged("decode_1b_fp8", nd=64, lo=128, hi=2048, np=0, qlo=0, qhi=0, chi=0, Hq=32, Hkv=8, D=64, kv="fp8"),
        # Long-context decode, 70B heads: the largest call.
        _paged("decode_70b_long", nd=128, lo=16384, hi=32768, np=0, qlo=0, qhi=0, chi=0, Hq=64, Hkv=8, D=128),
        # Prompt processing of an 8B model: eight ragged prompts.
        _paged("prefill_8b", nd=0, lo=0, hi=0, np=8, qlo=512, qhi=4096, chi=0, Hq=32, Hkv=8, D=128),
        # Continuous batching: 256 decodes and four 512-token prefill chunks.
        _paged("mixed_8b", nd=256, lo=256, hi=8192, log=True, np=4, qlo=512, qhi=512, chi=4096, Hq=32, Hkv=8, D=128),
        # QKV projection of a large decode batch.
        _qkv("qkv_decode_8b", n=256, hidden=4096, Hq=32, Hkv=8, D=128),
        # QKV projection of the eight prompts above.
        _qkv("qkv_prefill_8b", n=19679, hidden=4096, Hq=32, Hkv=8, D=128),
        # The op-level drop-in: a left-padded batch with the engine's bias.
        _dense("dense_1b", B=8, Tq=512, T=1024, Hq=32, Hkv=8, D=64),
    ]


def _layer(name, B, lo, hi, Hq, Hkv, D, dtype):
    return {"name": name, "kind": "layer", "B": B, "lo": lo, "hi": hi, "Hq": Hq, "Hkv": Hkv, "D": D,
            "dtype": dtype, "kv": dtype, "bs": 16}


def _forward(name, B, lo, hi, Hq, Hkv, D, dtype):
    return {**_layer(name, B, lo, hi, Hq, Hkv, D, dtype), "kind": "forward"}


def _paged(name, nd, lo, hi, np, qlo, qhi, chi, Hq, Hkv, D, dtype="bf16", kv=None, bs=16, log=False):
    return {"name": name, "kind": "paged", "nd": nd, "lo": lo, "hi": hi, "log": log, "np": np, "qlo": qlo,
            "qhi": qhi, "chi": chi, "Hq": Hq, "Hkv": Hkv, "D": D, "dtype": dtype, "kv": kv or dtype, "bs": bs}


def _qkv(name, n, hidden, Hq, Hkv, D, kv="bf16"):
    return {"name": name, "kind": "qkv", "n": n, "hidden": hidden, "Hq": Hq, "Hkv": Hkv, "D": D, "dtype": "bf16",
            "kv": kv, "bs": 16}


def _dense(name, B, Tq, T, Hq, Hkv, D, dtype="bf16"):
    return {"name": name, "kind": "dense", "B": B, "Tq": Tq, "T": T, "Hq": Hq, "Hkv": Hkv, "D": D, "dtype": dtype}


def _logint(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the listed ones' ranges, sizes spread over them."""
    heads = rng.choice([(32, 8, 64), (32, 8, 128), (64, 8, 128)])
    # an odd block size now and then: the engine's is a free setting
    bs = rng.choice([16, 16, 16, 8, 32, 24])
    f16 = rng.choice(["bf16", "bf16", "f16"])
    kind = rng.choice(["layer", "forward", "generic", "decode", "decode", "prefill", "mixed", "qkv", "qkv", "dense"])
    if kind == "layer":
        lo = _logint(rng, 8, 512)
        c = _layer("", _logint(rng, 1, 32), lo, 4 * lo, 32, 8, 64, rng.choice(["f32", "f32", "bf16"]))
    elif kind == "forward":
        lo = _logint(rng, 64, 1024)
        Hq, Hkv, D = rng.choice([(32, 8, 64), (32, 8, 128)])
        c = _forward("", _logint(rng, 1, 128), lo, 4 * lo, Hq, Hkv, D, f16)
    elif kind == "generic":
        # fp32 models, and 16-bit ones whose head dim is neither 64 nor 128
        dt, D = rng.choice([("f32", 64), ("f32", 64), ("f32", 128), ("bf16", 96), ("bf16", 80), ("f16", 256)])
        qlo = _logint(rng, 8, 512)
        np = _logint(rng, 1, 8)
        nd = rng.choice([0, 0, _logint(rng, 1, 16)])
        c = _paged("", nd, 64, 1024, np, qlo, 2 * qlo, rng.choice([0, 0, 512]), 32, 8, D, dt)
    elif kind == "decode":
        lo = _logint(rng, 64, 8192)
        Hq, Hkv, D = heads
        # at most a quarter million cached tokens
        nd = _logint(rng, 1, max(1, min(256, (1 << 18) // (2 * lo))))
        c = _paged("", nd, lo, 3 * lo, 0, 0, 0, 0, Hq, Hkv, D, f16, rng.choice([None, None, "fp8"]))
    elif kind == "prefill":
        qlo = _logint(rng, 16, 1024)
        Hq, Hkv, D = heads
        c = _paged("", 0, 0, 0, _logint(rng, 1, 8), qlo, 4 * qlo, rng.choice([0, 0, 1024]), Hq, Hkv, D, f16,
                   rng.choice([None, None, None, "fp8"]))
    elif kind == "mixed":
        lo = _logint(rng, 64, 1024)
        Hq, Hkv, D = heads
        qlo = _logint(rng, 16, 512)
        c = _paged("", _logint(rng, 8, 128), lo, 8 * lo, _logint(rng, 1, 4), qlo, 2 * qlo, 2048, Hq, Hkv, D, f16,
                   rng.choice([None, None, "fp8"]), log=True)
    elif kind == "qkv":
        hidden, Hq, Hkv, D = rng.choice([(2048, 32, 8, 64), (4096, 32, 8, 128), (4096, 32, 8, 128)])
        c = _qkv("", _logint(rng, 1, 16384), hidden, Hq, Hkv, D, rng.choice(["bf16", "bf16", "fp8"]))
    else:
        T = _logint(rng, 64, 2048)
        Hq, Hkv, D = heads
        c = _dense("", _logint(rng, 1, 8), rng.choice([T, max(1, T // 2), max(1, T // 5)]), T, Hq, Hkv, D, f16)
    del c["name"]
    if c["kind"] in ("layer", "paged"):
        c["bs"] = bs
    return c


# ------------------------------------------------------------------ lengths
def _lengths(case):
    """(context lengths, query lengths) of the batch, from the case alone."""
    g = torch.Generator().manual_seed(0)
    if case["kind"] in ("layer", "forward"):
        ctx = torch.randint(case["lo"], case["hi"] + 1, (case["B"],), generator=g).tolist()
        return ctx, [1] * case["B"]
    nd, lo, hi = case["nd"], case["lo"], case["hi"]
    if case["log"]:
        u = torch.rand(nd, generator=g, dtype=torch.float64).tolist()
        L = [int(round(math.exp(math.log(lo) + x * (math.log(hi) - math.log(lo))))) for x in u]
    else:
        L = torch.randint(lo, hi + 1, (nd,), generator=g).tolist()
    ctx, ql = [x - 1 for x in L], [1] * nd
    if case["np"]:
        ql += torch.randint(case["qlo"], case["qhi"] + 1, (case["np"],), generator=g).tolist()
        ctx += torch.randint(0, case["chi"] + 1, (case["np"],), generator=g).tolist()
    return ctx, ql


def _left_padded(case):
    """Key counts of a dense batch's sequences: at least one key per query row."""
    g = torch.Generator().manual_seed(0)
    return torch.randint(case["Tq"], case["T"] + 1, (case["B"],), generator=g).tolist()


# ------------------------------------------------------------------ inputs
class _Values:
    """N(0, 1) values drawn on the GPU from the seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def __call__(self, *shape, dtype, scale=1.0):
        n, out = math.prod(shape), torch.empty(shape, dtype=dtype, device="cuda")
        flat = out.view(-1)
        for o in range(0, n, 1 << 26):
            m = min(1 << 26, n - o)
            x = torch.randn(m, generator=self.g, device="cuda")
            flat[o:o + m] = (x * scale if scale != 1.0 else x).to(dtype)
        return out


def _rope_table(rows, D, dtype):
    ang = torch.arange(rows, device="cuda", dtype=torch.float64).unsqueeze(1) \
        * THETA ** (-2 * torch.arange(D // 2, device="cuda", dtype=torch.float64) / D)
    return torch.cos(ang).to(dtype), torch.sin(ang).to(dtype)


def _inputs(case, seed):
    """Tensors of a paged batch: pool, block table, new tokens, RoPE table."""
    ctx, ql = _lengths(case)
    L = [c + q for c, q in zip(ctx, ql)]
    dt, kv = DTYPES[case["dtype"]], DTYPES[case["kv"]]
    Hq, Hkv, D, bs = case["Hq"], case["Hkv"], case["D"], case["bs"]
    val = _Values(seed)
    need = [-(-x // bs) for x in L]
    nb = sum(need) + 1                                    # block 0 is the reserved one
    perm = (torch.randperm(nb - 1, generator=val.g, device="cuda") + 1).to(torch.int32)
    bt = torch.zeros(len(L), max(need), dtype=torch.int32, device="cuda")
    o = 0
    for i, n in enumerate(need):
        bt[i, :n] = perm[o:o + n]
        o += n
    rows = sum(ql)
    seq = torch.repeat_interleave(torch.arange(len(L)), torch.tensor(ql)).cuda()
    pos = torch.cat([torch.arange(c, c + q) for c, q in zip(ctx, ql)]).cuda()
    slots = bt[seq, pos // bs].to(torch.int64) * bs + pos % bs
    cos, sin = _rope_table(max(L), D, dt)
    s = {"ctx": ctx, "ql": ql, "L": L, "bt": bt, "pos": pos, "slots": slots, "cos": cos, "sin": sin,
         "k_cache": val(nb * bs, Hkv, D, dtype=kv), "v_cache": val(nb * bs, Hkv, D, dtype=kv)}
    if case["kind"] == "forward":
        hid = Hq * D
        s["x"] = val(len(L), 1, hid, dtype=dt)
        for n, h in (("q", Hq), ("k", Hkv), ("v", Hkv)):
            s["w" + n] = val(h * D, hid, dtype=dt, scale=hid ** -0.5)
        s["wo"] = val(hid, hid, dtype=dt, scale=hid ** -0.5)
    else:
        s["q"] = val(rows, Hq, D, dtype=dt)
        s["k"], s["v"] = val(rows, Hkv, D, dtype=dt), val(rows, Hkv, D, dtype=dt)
    return s


def _qkv_inputs(case, seed):
    val = _Values(seed)
    n, hid, D = case["n"], case["hidden"], case["D"]
    bf = DTYPES[case["dtype"]]
    s = {"x": val(n, hid, dtype=bf)}
    for w, h in (("q", case["Hq"]), ("k", case["Hkv"]), ("v", case["Hkv"])):
        s["w" + w] = val(h * D, hid, dtype=bf, scale=hid ** -0.5)
    ns = (-(-n // case["bs"]) + 1) * case["bs"]
    s["cos"], s["sin"] = _rope_table(8192, D, bf)
    s["pos"] = torch.randint(0, 8192, (n,), generator=val.g, device="cuda")
    s["slots"] = (torch.randperm(ns - case["bs"], generator=val.g, device="cuda") + case["bs"])[:n].contiguous()
    for c in ("k_cache", "v_cache"):
        s[c] = torch.zeros(ns, case["Hkv"], D, dtype=DTYPES[case["kv"]], device="cuda")
    return s


def _dense_inputs(case, seed):
    val = _Values(seed)
    B, Tq, T, D = case["B"], case["Tq"], case["T"], case["D"]
    dt = DTYPES[case["dtype"]]
    s = {"q": val(B, Tq, case["Hq"], D, dtype=dt), "k": val(B, T, case["Hkv"], D, dtype=dt),
         "v": val(B, T, case["Hkv"], D, dtype=dt)}
    # the engine's bias: 0 where key j of the left-padded window is one of the
    # sequence's and not after the query row's own position, else -inf
    j, r = torch.arange(T, device="cuda"), torch.arange(Tq, device="cuda")
    first = T - torch.tensor(_left_padded(case), device="cuda")
    seen = (j >= first[:, None, None]) & (j <= (T - Tq + r)[None, :, None])
    s["bias"] = torch.where(seen, 0.0, -math.inf).to(dt)
    return s


class _Config:
    def __init__(self, case):
        self.num_attn_heads, self.num_kv_heads, self.head_dim = case["Hq"], case["Hkv"], case["D"]
        self.hidden_size, self.dtype = case["Hq"] * case["D"], DTYPES[case["dtype"]]


def prepare(case, seed):
    """What the program holds before the call: inputs, weights, and the plan
    of the engine step (built once per step and used by every layer)."""
    if case["kind"] == "qkv":
        s = _qkv_inputs(case, seed)
        s["q_out"] = torch.empty(case["n"], case["Hq"], case["D"], dtype=s["x"].dtype, device="cuda")
    elif case["kind"] == "dense":
        s = _dense_inputs(case, seed)
    elif case["kind"] == "paged":
        s = _inputs(case, seed)
        s["plan"] = paged.AttentionPlan(s["ql"], s["L"], num_q_heads=case["Hq"], num_kv_heads=case["Hkv"],
                                        head_dim=case["D"], block_size=case["bs"], dtype=s["q"].dtype, device="cuda")
        s["out"] = torch.empty_like(s["q"])
    else:
        s = _inputs(case, seed)
        B, Hkv, D = case["B"], case["Hkv"], case["D"]
        pre = "model.layers.0.self_attn."
        w = {pre + n + "_proj.weight": s.get("w" + n, torch.zeros(1)) for n in "qkvo"}
        s["layer"] = gllm_amd.Attention(0, _Config(case), w)
        s["meta"] = gllm_amd.AttentionMetadata(
            query_lens=torch.ones(B, dtype=torch.int32, device="cuda"),
            seq_lens=torch.tensor(s["L"], dtype=torch.int32, device="cuda"), max_seq_len=max(s["L"]),
            block_table=s["bt"], slot_mapping=None, query_slot_mapping=s["slots"].view(B, 1), bias=None,
            block_size=case["bs"])
        s["cos_pos"], s["sin_pos"] = (s[c][s["pos"]].view(B, 1, D // 2) for c in ("cos", "sin"))
        s["pool"] = torch.stack([s.pop("k_cache"), s.pop("v_cache")])
        s["k_cache"], s["v_cache"] = s["pool"][0], s["pool"][1]
        if case["kind"] == "layer":
            for n, h in (("q", case["Hq"]), ("k", Hkv), ("v", Hkv)):
                s[n] = s[n].view(B, 1, h, D)
        # the step's first layer builds the plan; this call is another one
        gllm_amd.attention.plan_for(s["meta"], num_q_heads=case["Hq"], num_kv_heads=Hkv, head_dim=D,
                                    dtype=DTYPES[case["dtype"]], device=s["pool"].device)
    s["case"] = case
    return s


def run(s):
    kind = s["case"]["kind"]
    if kind == "dense":
        return gllm_amd.reference_attention(s["q"], s["k"], s["v"], s["bias"])
    if kind == "qkv":
        paged.qkv_rope_kv_write(s["x"], s["wq"], s["wk"], s["wv"], s["cos"], s["sin"], s["k_cache"], s["v_cache"],
                                s["slots"], q_out=s["q_out"], rope_rows=s["pos"])
        return s["q_out"], s["k_cache"], s["v_cache"]
    if kind == "layer":
        out = s["layer"].attention(s["q"], s["k"], s["v"], s["cos_pos"], s["sin_pos"], s["pool"], s["meta"])
    elif kind == "forward":
        out = s["layer"].forward(s["x"], s["cos_pos"], s["sin_pos"], s["pool"], s["meta"])
    else:
        rope = (s["cos"], s["sin"], "position")
        if paged.fused_kv_write_ok(s["plan"], s["k_cache"].dtype):
            out = paged.paged_attention(s["plan"], s["q"], s["k_cache"], s["v_cache"], s["bt"], out=s["out"],
                                        rope=rope, kv_new=(s["k"], s["v"]))
        else:
            paged.rope_kv_write(s["k"], s["v"], s["cos"], s["sin"], s["k_cache"], s["v_cache"], s["slots"],
                                rope_rows=s["pos"])
            out = paged.paged_attention(s["plan"], s["q"], s["k_cache"], s["v_cache"], s["bt"], out=s["out"],
                                        rope=rope)
    return out, s["k_cache"], s["v_cache"]


# ------------------------------------------------------------------ work
def work(case):
    e = SIZES[case["dtype"]]
    Hq, Hkv, D = case["Hq"], case["Hkv"], case["D"]
    if case["kind"] == "qkv":
        n, hid, cols = case["n"], case["hidden"], (Hq + 2 * Hkv) * D
        return {"bytes": (n * hid + cols * hid + n * Hq * D + n * D) * e + 2 * n * Hkv * D * SIZES[case["kv"]],
                "flops": 2 * n * hid * cols}
    if case["kind"] == "dense":
        B, Tq, T = case["B"], case["Tq"], case["T"]
        pairs = 0
        for L in _left_padded(case):          # visible (row, key) pairs
            pairs += sum(L - Tq + r + 1 for r in range(Tq))
        return {"bytes": (2 * B * Tq * Hq * D + 2 * B * T * Hkv * D + B * Tq * T) * e, "flops": 4 * Hq * D * pairs}
    ctx, ql = _lengths(case)
    rows = sum(ql)
    kv = 2 * Hkv * D * SIZES[case["kv"]]
    pairs = sum(q * c + q * (q + 1) // 2 for c, q in zip(ctx, ql))
    # cached K/V read, new K/V and q read, new K/V and the output written, RoPE rows, block ids
    nbytes = sum(ctx) * kv + rows * ((2 * Hkv + 2 * Hq) * D * e + D * e + kv) \
        + sum(-(-(c + q) // case["bs"]) for c, q in zip(ctx, ql)) * 4
    flops = 4 * Hq * D * pairs
    if case["kind"] == "forward":
        hid = Hq * D
        cols = (2 * Hq + 2 * Hkv) * D
        nbytes += hid * cols * e
        flops += 2 * rows * hid * cols
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------------------------------ accuracy
def tolerance(case):
    """About four times what the path is off the 64-bit result, whole outputs
    taken together: fp32 arithmetic, one rounding of 16-bit results (and of P
    and the rotated rows), one of an fp8 cache's new rows."""
    if case["dtype"] == "f32":
        return {"rel": 1e-5, "max": 2e-4}
    # one code of an fp8 row is an eighth of its value
    return {"rel": 1.5e-2, "max": 0.3 if case.get("kv") == "fp8" else 0.1}


def _rotate(x, c, s):
    h = x.shape[-1] // 2
    c, s = c.unsqueeze(-2), s.unsqueeze(-2)
    return torch.cat([x[..., :h] * c - x[..., h:] * s, x[..., :h] * s + x[..., h:] * c], -1)


def _softmax_v(q, k, v, hidden):
    """q [rows, Hq, D], k/v [keys, Hkv, D], hidden [rows, keys] -> [rows, Hq, D]."""
    rows, Hq, D = q.shape
    Hkv = k.shape[1]
    out = torch.empty_like(q)
    for h in range(Hkv):
        g = slice(h * (Hq // Hkv), (h + 1) * (Hq // Hkv))
        kh, vh = k[:, h].contiguous(), v[:, h].contiguous()
        for r in range(0, rows, 1024):
            sc = q[r:r + 1024, g].reshape(-1, D) @ kh.t().contiguous() / math.sqrt(D)
            sc = sc.view(-1, Hq // Hkv, kh.shape[0]).masked_fill(hidden[r:r + 1024].unsqueeze(1), -math.inf)
            p = torch.softmax(sc, -1).view(-1, kh.shape[0])
            out[r:r + 1024, g] = (p @ vh).view(-1, Hq // Hkv, D)
    return out


# a pool of more elements than this has no 64-bit copy beside it
_POOL = 1 << 30


def exact(case, seed):
    f = torch.float64
    Hq, Hkv, D = case["Hq"], case["Hkv"], case["D"]
    if case["kind"] == "dense":
        s = _dense_inputs(case, seed)
        q, k, v = (s[n].to(f) for n in "qkv")
        hidden = torch.isinf(s["bias"])
        return torch.stack([_softmax_v(q[b], k[b], v[b], hidden[b]) for b in range(case["B"])])
    if case["kind"] == "qkv":
        s = _qkv_inputs(case, seed)
        x = s["x"].to(f)
        cos, sin = s["cos"].to(f)[s["pos"]], s["sin"].to(f)[s["pos"]]
        q, k, v = ((x @ s["w" + n].to(f).t().contiguous()).view(-1, h, D) for n, h in (("q", Hq), ("k", Hkv), ("v", Hkv)))
        kc, vc = s["k_cache"].to(f), s["v_cache"].to(f)
        kc[s["slots"]], vc[s["slots"]] = _rotate(k, cos, sin), v
        return _rotate(q, cos, sin), kc, vc
    s = _inputs(case, seed)
    ctx, ql, bs = s["ctx"], s["ql"], case["bs"]
    cos, sin = s["cos"].to(f)[s["pos"]], s["sin"].to(f)[s["pos"]]
    if case["kind"] == "forward":
        x = s["x"].to(f).view(len(ql), -1)
        q, k, v = ((x @ s["w" + n].to(f).t().contiguous()).view(-1, h, D) for n, h in (("q", Hq), ("k", Hkv), ("v", Hkv)))
    else:
        q, k, v = (s[n].to(f) for n in "qkv")
    q, k = _rotate(q, cos, sin), _rotate(k, cos, sin)
    out = torch.empty_like(q)
    row = 0
    for i, (c, n) in enumerate(zip(ctx, ql)):
        p = torch.arange(c, device="cuda")
        slot = s["bt"][i, p // bs].to(torch.int64) * bs + p % bs
        ki, vi = (torch.cat([s[t][slot].to(f), new[row:row + n]]) for t, new in (("k_cache", k), ("v_cache", v)))
        r = torch.arange(n, device="cuda")
        hidden = torch.arange(c + n, device="cuda")[None, :] > (c + r)[:, None]
        out[row:row + n] = _softmax_v(q[row:row + n], ki, vi, hidden)
        row += n
    kc = vc = None
    if s["k_cache"].numel() <= _POOL:
        kc, vc = s["k_cache"].to(f), s["v_cache"].to(f)
        kc[s["slots"]], vc[s["slots"]] = k, v
    if case["kind"] == "forward":
        return (out.view(len(ql), -1) @ s["wo"].to(f).t().contiguous()).view(len(ql), 1, -1), kc, vc
    if case["kind"] == "layer":
        out = out.view(len(ql), 1, Hq, D)
    return out, kc, vc
