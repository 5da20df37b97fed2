"""The work that a user of this framework has it do, as cases that can be timed and compared.

Two kinds of case, each through the public entry points (`HipBackend`):

- "step": one forward pass's KV path, as an engine runs it: `begin_pass` with the pass's
  metadata, then per layer the attention call. Decode (one row per sequence), verify (a few
  rows per sequence) and prefill (a chunk of rows per sequence), on a binary16 or an f32
  arena, with or without sliding-window layers and shared prompt prefixes. "qkv" cases call
  `attention` (`Backend::attention`: q/k norm, RoPE, K/V store, attend); the others hand over
  finished q, k, v (`attend_append`). The arena already holds the sequences' earlier tokens;
  page tables are scattered over the pool as the allocator leaves them after some use.
- "proj": the step after attention: a bf16 weight product over the pass's rows
  (`matmul_bf16`), and with "vocab" the logits of those rows and their greedy pick
  (`argmax_rows`).

Head counts, page sizes, chunk and window sizes are those of the benchmark's configurations
and of the engine's defaults (pages of 128, chunks of up to 512 rows, 8 decode rows, window
2048 with every 4th or 8th layer full). All cases of a process share one context (one stream),
as an engine's passes do.
"""

from __future__ import annotations

import ctypes
import math
import random

import numpy as np
import torch

from yaxus_amd.backend import DeviceTensor, HipBackend
from yaxus_amd.kv import PassMeta

D = 128
EPS = 1e-6
THETA = 10000.0


def _step(name, batch, rows, ctx_lo, ctx_hi, **kw):
    """`rows` new tokens for each of `batch` sequences whose earlier lengths lie between
    ctx_lo and ctx_hi (evenly over their logarithm)."""
    c = dict(name=name, kind="step", batch=batch, rows=rows, ctx_lo=ctx_lo, ctx_hi=ctx_hi,
             prefix=0, hq=16, hkv=4, page=16, f32=False, qkv=True, layers=24, window=0,
             full_every=1, spread=1)
    c.update(kw)
    return c


def listed():
    return [
        # One user's chat turn: a single sequence, every layer a small launch.
        _step("decode_one", 1, 1, 600, 600, hq=24, page=128),
        # The headline of bench.py: 16 sequences of 4096 tokens.
        _step("decode_16x4096", 16, 1, 4095, 4095, qkv=False),
        # A server's mixed batch: many sequences of very different lengths.
        _step("decode_ragged", 48, 1, 60, 12000, hq=24, page=128, layers=8),
        # Long contexts on a model with sliding-window layers: 1 full + 3 window-2048.
        _step("decode_window", 4, 1, 32767, 32767, qkv=False, layers=8, window=2048, full_every=4),
        # Forks of one prompt: 16 sequences sharing its first 1024 tokens.
        _step("decode_forks", 16, 1, 1536, 4096, prefix=1024),
        # Speculative verification: 5 rows per sequence over a shared prompt of 2048 tokens.
        _step("verify_forks", 16, 5, 4091, 4091, prefix=2048),
        # Chunked prefill of 16 prompts at once.
        _step("prefill_chunks", 16, 256, 8, 2040, layers=6),
        # One long document, the engine's 512-row chunk, window layers with one full in 8.
        _step("prefill_long", 1, 512, 24000, 24000, hq=24, page=128, layers=8, window=2048, full_every=8),
        # The reference's own K/V precision: the engine's default of 8 decode rows.
        _step("decode_f32", 8, 1, 500, 8000, hq=24, page=128, f32=True, layers=12),
        # And its prompts.
        _step("prefill_f32", 4, 256, 100, 4000, page=128, f32=True, layers=3),
        # After the last layer of a 16-row decode pass: o_proj, the logits and the greedy pick.
        dict(name="head_16", kind="proj", t=16, k=2048, n=2048, vocab=151936),
        # o_proj over a prefill pass.
        dict(name="proj_4096", kind="proj", t=4096, k=2048, n=2048, vocab=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["decode", "decode", "verify", "prefill", "prefill", "proj", "head"])
    if what == "proj":
        t = _log(rng, 20, 4096)
        k, n = rng.choice([(2048, 2048), (3072, 2048), (2048, 3072), (1536, 2000)])
        return dict(kind="proj", t=t, k=k, n=n, vocab=0)
    if what == "head":
        return dict(kind="proj", t=_log(rng, 1, 80), k=2048, n=2048, vocab=_log(rng, 32000, 151936))
    hq, hkv = rng.choice([(16, 4), (24, 4), (32, 8), (16, 8)])
    c = dict(hq=hq, hkv=hkv, page=rng.choice([16, 128]), f32=rng.random() < 0.3,
             qkv=rng.random() < 0.6, spread=rng.randrange(1, 1000))
    if rng.random() < 0.25:
        c.update(window=rng.choice([1024, 2048]), full_every=rng.choice([4, 8]))
    if what == "prefill":
        c["batch"] = _log(rng, 1, 16)
        c["rows"] = min(_log(rng, 24, 512), 4096 // c["batch"])
        lo = _log(rng, 8, 3000)
        c.update(ctx_lo=lo, ctx_hi=min(_log(rng, lo, 24000), 40000 // c["batch"] + lo))
    else:
        c["batch"] = _log(rng, 1, 48)
        c["rows"] = 1 if what == "decode" else rng.randint(2, 8)
        lo = _log(rng, 50, 4000)
        c.update(ctx_lo=lo, ctx_hi=min(_log(rng, lo, 30000), 100000 // c["batch"] + lo))
        if rng.random() < 0.3:
            c["prefix"] = c["ctx_lo"] // 128 * 128
    c = _step("", c.pop("batch"), c.pop("rows"), c.pop("ctx_lo"), c.pop("ctx_hi"), **c)
    del c["name"]
    # As many layers as keep the pass within the largest listed one.
    c["layers"] = 1
    w = work(c)
    c["layers"] = max(1, min(24, int(min(2.5e9 / w["bytes"], 1.5e11 / w["flops"]))))
    return c


def _lengths(case):
    """The sequences' earlier lengths (tokens already in the arena)."""
    r = random.Random(case["spread"])
    lo, hi = case["ctx_lo"], case["ctx_hi"]
    return [min(hi, max(lo, _log(r, lo, hi))) if hi > lo else lo for _ in range(case["batch"])]


def _window(case, layer):
    return 0 if (layer + 1) % case["full_every"] == 0 else case["window"]


def work(case):
    if case["kind"] == "proj":
        t, k, n, v = case["t"], case["k"], case["n"], case["vocab"]
        b = 4 * t * k + 2 * n * k + 4 * t * n
        f = 2 * t * k * n
        if v:
            b += 2 * v * k + 4 * t * v + 4 * t
            f += 2 * t * k * v
        return {"bytes": b, "flops": f}
    hq, hkv, n, pre = case["hq"], case["hkv"], case["rows"], case["prefix"]
    size = 4 if case["f32"] else 2
    b = f = 0
    for layer in range(case["layers"]):
        w = _window(case, layer)
        keys = 0
        shared_from = pre
        for ctx in _lengths(case):
            first = max(0, ctx + 1 - w) if w else 0
            keys += ctx - max(first, pre) if ctx > max(first, pre) else 0
            shared_from = min(shared_from, first)
            for i in range(n):
                p = ctx + i + 1
                f += 4 * D * hq * (min(p, w) if w else p)
        keys += max(0, pre - shared_from)
        rows = case["batch"] * n
        b += keys * hkv * D * 2 * size          # K/V read
        b += rows * hkv * D * 2 * (size + 4)    # new K/V in, stored
        b += rows * hq * D * 4 * 2              # q in, output
    return {"bytes": b, "flops": f}


def tolerance(case):
    # Sums in f32: 1.4e-7 to 1.0e-6 from 64 bits. A binary16 arena whose new keys are
    # normalised and rotated on the way in: an f32 result in another order now and then
    # rounds to the neighbouring binary16 (up to 5.4e-6, in a short context one row's
    # output by about 2^-11 of a key's share).
    if case["kind"] == "step" and case["qkv"] and not case["f32"]:
        return {"rel": 2e-5, "max": 1e-2}
    return {"rel": 4e-6, "max": 1e-4}


_hip = None


def _backend():
    global _hip
    if _hip is None:
        _hip = HipBackend(0)
    return _hip


class _Torch(DeviceTensor):
    """A torch tensor as the backend's operand."""

    def __init__(self, t, dtype=np.float32):
        self.t, self.shape, self.dtype = t, tuple(t.shape), np.dtype(dtype)
        self.nbytes = t.numel() * t.element_size()
        self.ptr = ctypes.c_void_p(t.data_ptr())


class _View:
    """One layer's K (which = 0) or V (1) arena, for torch; it holds the arena."""

    def __init__(self, arena, layer, which):
        self.arena, kv = arena, arena.kv
        size = 4 if kv.f32 else 2
        self.__cuda_array_interface__ = dict(data=(kv.layer_ptr(layer, which).value, False),
                                             shape=(kv.pages * kv.page_bytes // size,),
                                             typestr="<f%d" % size, version=2)


class _Arena:
    """The KV arena of one state, destroyed once neither the state nor an output needs it."""

    def __init__(self, hip, *args, **kw):
        self.kv = hip.new_kv(*args, **kw)

    def view(self, layer, which):
        t = torch.as_tensor(_View(self, layer, which), device="cuda")
        t.arena = self  # an output outlives its state
        return t

    def __del__(self):
        self.kv.destroy()


def _gen(seed, what):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000003 + what)
    return g


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _layer_inputs(case, seed, layer):
    """(old K, old V, the pass's new inputs) of one layer. Old rows: the shared prefix, then
    each sequence's own tokens."""
    g = _gen(seed, layer)
    old = case["prefix"] + sum(n - case["prefix"] for n in _lengths(case))
    rows, hq, hkv = case["batch"] * case["rows"], case["hq"], case["hkv"]
    k, v = _normal(g, old, hkv, D), _normal(g, old, hkv, D)
    if case["qkv"]:
        new = (_normal(g, rows, (hq + 2 * hkv) * D), 0.1 * _normal(g, D), 0.1 * _normal(g, D))
    else:
        new = (_normal(g, rows, hkv, D), _normal(g, rows, hkv, D), _normal(g, rows, hq, D))
    return k, v, new


def _rope(case):
    """cos, sin of every position: [2][positions][64] f32 (f32 angles)."""
    i = torch.arange(0, D, 2, dtype=torch.float32, device="cuda")
    freq = 1.0 / torch.pow(torch.tensor(THETA, device="cuda"), i / D)
    n = max(_lengths(case)) + case["rows"]
    a = (torch.arange(n, dtype=torch.float32, device="cuda")[:, None] * freq[None, :]).double()
    return torch.stack([a.cos(), a.sin()]).float().contiguous()


def _metas(case, seed):
    """(pool pages, the pass that brings the arena to its state, the measured pass)."""
    page, n, pre = case["page"], case["rows"], case["prefix"]
    lens = _lengths(case)
    shared = pre // page
    need = [-(-(ctx + n) // page) for ctx in lens]
    pool = shared + sum(p - shared for p in need)
    pool += pool // 8
    ids = np.random.RandomState(seed % (1 << 31)).permutation(pool).astype(np.uint32)
    head, at = ids[:shared], shared
    tables = []
    for p in need:
        tables.append(np.concatenate([head, ids[at:at + p - shared]]))
        at += p - shared

    def meta(tables, spans):
        pos, slot, off, o = [], [], [], 0
        for t, (a, b) in zip(tables, spans):
            p = np.arange(a, b, dtype=np.uint32)
            pos.append(p)
            slot.append(t[p // page] * np.uint32(page) + p % np.uint32(page))
            off.append(np.full(b - a, o, np.uint32))
            o += len(t)
        pos = np.concatenate(pos)
        return PassMeta(ids=np.zeros(len(pos), np.uint32), pos=pos, kv_slot=np.concatenate(slot),
                        pt_off=np.concatenate(off), pages=np.concatenate(tables))

    fill_t = ([head] if pre else []) + [t for t, c in zip(tables, lens) if c > pre]
    fill_s = ([(0, pre)] if pre else []) + [(pre, c) for c in lens if c > pre]
    return pool, meta(fill_t, fill_s), meta(tables, [(c, c + n) for c in lens])


def prepare(case, seed):
    hip = _backend()
    if case["kind"] == "proj":
        return _prepare_proj(case, seed)
    pool, fill, meta = _metas(case, seed)
    rows, hq, hkv, layers = case["batch"] * case["rows"], case["hq"], case["hkv"], case["layers"]
    arena = _Arena(hip, layers, pool, case["page"], hkv, D, f32=case["f32"])
    hip.begin_pass(fill)
    new = []
    for layer in range(layers):
        k, v, x = _layer_inputs(case, seed, layer)
        torch.cuda.synchronize()
        hip.append(arena.kv, layer, _Torch(k), _Torch(v))
        hip.sync()
        new.append([_Torch(t) for t in x])
        del k, v
    out = torch.empty(layers, rows, hq * D, device="cuda", dtype=torch.float32)
    rope = _Torch(_rope(case)) if case["qkv"] else None
    torch.cuda.synchronize()
    return dict(case=case, arena=arena, meta=meta, new=new, rope=rope, out=out,
                outs=[_Torch(out[i]) for i in range(layers)], stored=(arena.view(0, 0), arena.view(0, 1)),
                windows=[_window(case, i) for i in range(layers)])


def _bf16(x):
    return x.to(torch.bfloat16)


def _proj_inputs(case, seed):
    g = _gen(seed, 0)
    k, n, t, v = case["k"], case["n"], case["t"], case["vocab"]
    x = _normal(g, t, k)
    w = _bf16(_normal(g, n, k) / math.sqrt(k))
    if not v:
        return x, w, None, None
    return x, w, _normal(g, t, k), _bf16(_normal(g, v, k) / math.sqrt(k))


def _prepare_proj(case, seed):
    x, w, h, u = _proj_inputs(case, seed)
    t, n, v = case["t"], case["n"], case["vocab"]
    s = dict(case=case, x=_Torch(x), w=_Torch(w, np.uint16),
             out=_Torch(torch.empty(t, n, device="cuda", dtype=torch.float32)))
    if v:
        s.update(h=_Torch(h), u=_Torch(u, np.uint16),
                 logits=_Torch(torch.empty(t, v, device="cuda", dtype=torch.float32)),
                 picks=_Torch(torch.empty(t, device="cuda", dtype=torch.int32), np.uint32))
    torch.cuda.synchronize()
    return s


def run(s):
    hip, case = _hip, s["case"]
    if case["kind"] == "proj":
        hip.matmul_bf16(s["x"], s["w"], out=s["out"])
        if not case["vocab"]:
            return {"out": s["out"].t}
        hip.matmul_bf16(s["h"], s["u"], out=s["logits"])
        hip.argmax_rows(s["logits"], out=s["picks"])
        return {"out": s["out"].t, "logits": s["logits"].t, "picks": s["picks"].t}
    kv, hq = s["arena"].kv, case["hq"]
    hip.begin_pass(s["meta"])
    for layer, (x, out, w) in enumerate(zip(s["new"], s["outs"], s["windows"])):
        if case["qkv"]:
            hip.attention(kv, layer, x[0], x[1], x[2], s["rope"], EPS, hq, window=w, out=out)
        else:
            hip.attend_append(kv, layer, x[0], x[1], x[2], hq, window=w, out=out)
    return {"out": s["out"], "stored_k": s["stored"][0], "stored_v": s["stored"][1]}


def _norm_rope(x, w, cos, sin):
    """RMSNorm (weight offset 1) and half-split RoPE of x [rows][heads][D], f64."""
    y = x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * (1.0 + w.double())
    a, b = y[..., :D // 2], y[..., D // 2:]
    c, s = cos[:, None, :], sin[:, None, :]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def exact(case, seed):
    if case["kind"] == "proj":
        x, w, h, u = _proj_inputs(case, seed)
        got = {"out": x.double() @ w.double().t().contiguous()}
        if u is not None:
            got["logits"] = torch.cat([h.double() @ p.double().t().contiguous() for p in u.split(16384)], 1)
            got["picks"] = None
        return got
    hq, hkv, n, pre = case["hq"], case["hkv"], case["rows"], case["prefix"]
    G = hq // hkv
    lens = _lengths(case)
    rope = _rope(case).double() if case["qkv"] else None
    stored = (lambda t: t.float().double()) if case["f32"] else (lambda t: t.float().half().double())
    out = torch.empty(case["layers"], case["batch"] * n, hq, D, device="cuda", dtype=torch.float64)
    for layer in range(case["layers"]):
        ok, ov, new = _layer_inputs(case, seed, layer)
        ok, ov = stored(ok), stored(ov)
        w, at = _window(case, layer), pre
        for i, ctx in enumerate(lens):
            r = slice(i * n, i * n + n)
            own = slice(at, at + ctx - pre)
            at += ctx - pre
            if case["qkv"]:
                x = new[0][r].double().view(n, hq + 2 * hkv, D)
                cos, sin = rope[0, ctx:ctx + n], rope[1, ctx:ctx + n]
                q = _norm_rope(x[:, :hq], new[1], cos, sin)
                nk, nv = _norm_rope(x[:, hq:hq + hkv], new[2], cos, sin), x[:, hq + hkv:]
            else:
                nk, nv, q = (t[r].double() for t in new)
            k = torch.cat([ok[:pre], ok[own], stored(nk)])
            v = torch.cat([ov[:pre], ov[own], stored(nv)])
            first = max(0, ctx + 1 - w) if w else 0
            pos = torch.arange(first, ctx + n, device="cuda")
            row = torch.arange(ctx, ctx + n, device="cuda")[:, None]
            seen = pos[None, :] <= row
            if w:
                seen &= pos[None, :] > row - w
            seen = seen.repeat_interleave(G, 0)
            for h in range(hkv):
                qh = q[:, h * G:(h + 1) * G].reshape(n * G, D)
                score = qh @ k[first:, h].t().contiguous() / math.sqrt(D)
                p = score.masked_fill(~seen, -math.inf).softmax(-1)
                out[layer, r, h * G:(h + 1) * G] = (p @ v[first:, h].contiguous()).view(n, G, D)
                del score, p
    return {"out": out.view(case["layers"], -1, hq * D), "stored_k": None, "stored_v": None}
