"""What a user of this library has it do, as cases that can be timed and checked.

The engine around the library (24 query heads over 4 kv-heads; 256-dim heads in its real model,
128-dim heads in its benchmark geometry) makes three kinds of call:

  attend    the attention alone: decode (1 row per stream), speculative verify (2 .. 16 rows) and
            prompt chunks (17 .. 2048 rows), over f16 or q8_0 caches held as one range of cells
            per stream or as shuffled 256-cell pages, with the lengths as the mask or with
            llama.cpp's f16 mask handed over
  layer     a whole full-attention layer step around it: norm + RoPE + K/V store, then the
            attention with the output gate fused
  gdn       the recurrent state of a linear-attention layer over a verify block or a prompt chunk

Every case is one public call (two for `layer`) as an engine makes it, on inputs that are on the
GPU already, with the handle and its workspace kept from call to call.
"""
from __future__ import annotations

import math
import pathlib
import sys

import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parents[1] / "sixi-asi_amd"))

import sixi_attn as sa  # noqa: E402

H, HKV = 24, 4          # query heads and kv-heads of the engine's model
GDN_GROUPS, GDN_DIM = 48, 128   # value heads and state size of its linear-attention layers
PAGE = 256
EPS, ROPE_BASE, N_ROT = 1e-6, 1e7, 64


def _attend(name, streams, rows, lo, hi, dim, kv, layout="cells", mask="lengths", ragged=False):
    return {"name": name, "kind": "attend", "streams": streams, "rows": rows, "cached_lo": lo, "cached_hi": hi,
            "dim": dim, "kv": kv, "layout": layout, "mask": mask, "ragged": ragged}


def listed():
    return [
        # one user, one token at a time: the smallest call, latency and launches
        _attend("decode_one", 1, 1, 4095, 4095, 256, "f16"),
        # one user's drafted block through the ggml hook, which hands llama.cpp's mask over
        _attend("verify_one_mask", 1, 9, 8003, 8003, 128, "f16", mask="llama"),
        # a full server verifying 16-token drafts out of the page pool, contexts of 0.5k to 16k
        _attend("verify_batch_paged", 32, 16, 512, 15873, 128, "f16", layout="paged"),
        # the engine's operating point, short drafts for every slot: f16 and q8_0 caches
        _attend("verify_short_f16", 32, 4, 512, 15873, 256, "f16"),
        _attend("verify_short_q8", 32, 6, 512, 15873, 256, "q8_0", layout="paged"),
        # a few long documents over a q8_0 cache
        _attend("long_verify_q8", 8, 8, 40000, 50000, 128, "q8_0"),
        # a prompt's middle chunk at both head sizes
        _attend("prefill_chunk_256", 1, 2048, 2048, 2048, 256, "f16"),
        _attend("prefill_chunk_128", 1, 2048, 4096, 4096, 128, "f16", layout="paged"),
        # the next turn of a chat: a short prompt behind a long cached context
        _attend("chat_turn_q8", 1, 173, 11400, 11400, 256, "q8_0"),
        # a layer step of a half-full server with ragged drafts, pages, gated output
        {"name": "layer_step", "kind": "layer", "streams": 12, "rows": 7, "cached_lo": 300, "cached_hi": 9000,
         "ragged": True},
        # the linear-attention layer of the full verify batch, and of one user's prompt chunk
        {"name": "gdn_verify_batch", "kind": "gdn", "streams": 32, "rows": 16, "ragged": False, "decay_first": True},
        {"name": "gdn_chunk", "kind": "gdn", "streams": 1, "rows": 2048, "ragged": False, "decay_first": True},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


MAX_BYTES, MAX_FLOPS = 6.0e8, 1.25e11  # within the largest listed cases


def draw(rng):
    kind = rng.choice(("step", "step", "step", "chunk", "chunk", "layer", "gdn"))
    if kind == "gdn":
        if rng.random() < 0.3:
            return {"kind": "gdn", "streams": 1, "rows": _log_int(rng, 17, 2000), "ragged": False, "decay_first": True}
        return {"kind": "gdn", "streams": _log_int(rng, 1, 31), "rows": rng.randint(1, 16),
                "ragged": rng.random() < 0.5, "decay_first": rng.random() < 0.75}
    if kind == "layer":
        hi = _log_int(rng, 300, 12000)
        case = {"kind": "layer", "streams": _log_int(rng, 1, 32), "rows": rng.randint(1, 16),
                "cached_lo": _log_int(rng, 100, hi), "cached_hi": hi, "ragged": rng.random() < 0.7}
    else:
        if kind == "step":
            streams, rows = _log_int(rng, 1, 32), rng.randint(1, 16)
            hi = _log_int(rng, 256, 16384 if streams > 8 else 50000)
        else:
            streams, rows = rng.choice((1, 1, 1, 2, 4)), _log_int(rng, 17, 2048)
            hi = _log_int(rng, 64, 30000)
        lo = max(1, int(hi * rng.uniform(0.1, 1.0))) if streams > 1 else hi
        layout = rng.choice(("cells", "paged"))
        mask = "llama" if layout == "cells" and rng.random() < 0.3 else "lengths"
        case = _attend("", streams, rows, lo, hi, rng.choice((128, 256)), rng.choice(("f16", "f16", "q8_0")), layout,
                       mask, streams > 1 and rng.random() < 0.5)
        del case["name"]
    while work(case)["bytes"] > MAX_BYTES or work(case)["flops"] > MAX_FLOPS:
        case["cached_hi"] = max(16, int(case["cached_hi"] * 0.8))
        case["cached_lo"] = min(case["cached_lo"], case["cached_hi"])
        if case["cached_hi"] <= 4096 and case["rows"] > 16:
            case["rows"] = max(17, int(case["rows"] * 0.9))
    return case


# ---- sizes ----

def _spread(n, lo, hi):
    """n values over [lo, hi], both ends among them, in no order (a fixed shuffle by a step coprime to n)."""
    if n == 1:
        return [hi]
    step = next(k for k in range(n // 2 + 1, 2 * n) if math.gcd(k, n) == 1)
    return [lo + (hi - lo) * (i * step % n) // (n - 1) for i in range(n)]


def _lengths(case):
    """(cached cells, block rows) of each stream."""
    cached = _spread(case["streams"], case.get("cached_lo", 0), case.get("cached_hi", 0))
    rows = [case["rows"]] * case["streams"]
    if case["ragged"]:
        rows = _spread(case["streams"], (case["rows"] + 1) // 2, case["rows"])[::-1]
    return cached, rows


def _dim(case):
    return case.get("dim", 256)


def _row_bytes(case):
    return _dim(case) // 32 * 34 if case.get("kv") == "q8_0" else 2 * _dim(case)


def work(case):
    cached, rows = _lengths(case)
    n = sum(rows)
    if case["kind"] == "gdn":
        state = case["streams"] * GDN_GROUPS * GDN_DIM * GDN_DIM
        return {"bytes": 2 * 4 * state + n * GDN_GROUPS * 4 * (4 * GDN_DIM + 2),
                "flops": 6 * GDN_DIM * GDN_DIM * GDN_GROUPS * n}
    d = _dim(case)
    flops = 4 * d * H * sum(r * c + r * (r + 1) // 2 for c, r in zip(cached, rows))
    out = n * H * d * 4
    if case["kind"] == "layer":
        # q and gate, k and v read once; the cached cells read, the new cells written; out written
        return {"bytes": n * (2 * H * d * 4 + 2 * HKV * d * 4) + 2 * HKV * d * 2 * (sum(cached) + n) + out,
                "flops": flops}
    q = n * H * d * (2 if _half_q(case) else 4)
    return {"bytes": 2 * HKV * _row_bytes(case) * sum(c + r for c, r in zip(cached, rows)) + q + out, "flops": flops}


def _half_q(case):
    """The layer before hands f16 queries over an f16 cache, f32 ones over q8_0 (ggml quantises them from f32)."""
    return case["kind"] == "layer" or (case["rows"] > 16 and case["kv"] == "f16")


# ---- inputs ----

def _cells(gen, shape, kv):
    """Cache rows: f16 values, or q8_0 blocks {f16 scale; 32 int8} of such values."""
    x = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float16)
    if kv == "f16":
        return x
    b = x.reshape(*shape[:-1], shape[-1] // 32, 32).float()
    d = b.abs().amax(-1, keepdim=True) / 127
    q = torch.round(b / d).clamp_(-127, 127).to(torch.int8).view(torch.uint8)
    return torch.cat([d.half().view(torch.uint8), q], dim=-1).reshape(*shape[:-1], -1)


def _caches(gen, case, cached, rows):
    """K and V as the engine holds them and, paged, the table: [streams, capacity, kv-heads, row] or pages
    [n, 256, kv-heads, row] whose kv-heads lie one after the other, at shuffled places."""
    kv, d, s = case.get("kv", "f16"), _dim(case), case["streams"]
    pages = [-(-(c + r) // PAGE) for c, r in zip(cached, rows)]
    if case["kind"] == "layer" or case["layout"] == "paged":
        n = sum(pages)
        k, v = (_cells(gen, (n, HKV, PAGE, d), kv).permute(0, 2, 1, 3) for _ in range(2))
        order = torch.randperm(n, generator=gen, device="cuda").to(torch.int32)
        table = torch.zeros((s, max(pages)), dtype=torch.int32, device="cuda")
        at = 0
        for i, p in enumerate(pages):
            table[i, :p] = order[at:at + p]
            at += p
        return k, v, table
    cap = max(pages) * PAGE
    k, v = (_cells(gen, (s, cap, HKV, d), kv) for _ in range(2))
    return k, v, None


def _i32(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


def _llama_mask(cached, rows, n_rows, n_cells):
    """llama.cpp's f16 mask of the block: row j of a stream sees its cells 0 .. cached + j."""
    last = (_i32(cached)[:, None] + torch.arange(n_rows, device="cuda"))[:, :, None]
    seen = torch.arange(n_cells, device="cuda") <= last
    seen &= (torch.arange(n_rows, device="cuda") < _i32(rows)[:, None])[:, :, None]
    return torch.where(seen, 0.0, -math.inf).to(torch.float16)[:, None]


def _inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    cached, rows = _lengths(case)
    s, n_rows = case["streams"], case["rows"]

    def randn(*shape):
        return torch.randn(shape, generator=gen, device="cuda")

    if case["kind"] == "gdn":
        g, d = GDN_GROUPS, GDN_DIM
        unit = torch.nn.functional.normalize
        st = {"q": unit(randn(s, n_rows, g, d), dim=-1) / d ** 0.5, "k": unit(randn(s, n_rows, g, d), dim=-1),
              "v": randn(s, n_rows, g, d), "state": randn(s, g, d, d) * 0.3,
              # decays of exp(-softplus) gates: mostly close to 1, a few forgetting quickly
              "alpha": torch.exp(-0.1 * torch.nn.functional.softplus(1.5 * randn(s, n_rows, g))),
              "beta": torch.sigmoid(randn(s, n_rows, g)),
              "q_len": _i32(rows) if case["ragged"] else None,
              # the accepted part of each drafted block; a prompt chunk is kept whole
              "snap": _i32([(r + i % 3) // 2 for i, r in enumerate(rows)]) if n_rows <= 16 else None}
        return st
    d = _dim(case)
    k, v, table = _caches(gen, case, cached, rows)
    st = {"k": k, "v": v, "table": table, "kv_len": _i32(cached), "q_len": _i32(rows)}
    if case["kind"] == "layer":
        st.update(qg=randn(s, n_rows, H, 2 * d), k_new=randn(s, n_rows, HKV, d), v_new=randn(s, n_rows, HKV, d),
                  q_norm=1.0 + 0.2 * randn(d), k_norm=1.0 + 0.2 * randn(d))
        return st
    st["q"] = 2.0 * randn(s, n_rows, H, d)
    if _half_q(case):
        st["q"] = st["q"].half()
    if case["mask"] == "llama":
        st["mask"] = _llama_mask(cached, rows, n_rows, k.shape[1])
    return st


def prepare(case, seed):
    st = _inputs(case, seed)
    st["case"] = case
    s, n_rows = case["streams"], case["rows"]
    if case["kind"] == "gdn":
        st["y"] = torch.zeros_like(st["v"])
        st["state_out"] = torch.empty_like(st["state"])
        return st
    d = _dim(case)
    st["fa"] = sa.FlashAttnExt()
    st["out"] = torch.zeros((s, n_rows, H, d), dtype=torch.float32, device="cuda")
    if case["kind"] == "layer":
        st["q"] = torch.zeros((s, n_rows, H, d), dtype=torch.float16, device="cuda")
    return st


# ---- one pass ----

def run(st):
    case = st["case"]
    if case["kind"] == "gdn":
        sa.gdn_verify(st["q"], st["k"], st["v"], st["alpha"], st["beta"], st["y"], st["state"], st["state_out"],
                      q_len=st["q_len"], snap=st["snap"], decay_first=case["decay_first"])
        return {"y": st["y"], "state": st["state_out"]}
    if case["kind"] == "layer":
        sa.qk_prologue(st["qg"], st["k_new"], st["v_new"], st["q_norm"], st["k_norm"], st["q"], st["k"], st["v"],
                       st["kv_len"], st["q_len"], eps=EPS, rope_base=ROPE_BASE, n_rot=N_ROT, page_table=st["table"])
        st["fa"](st["q"], st["k"], st["v"], st["out"], kv_len=st["kv_len"], q_len=st["q_len"],
                 page_table=st["table"], gate=st["qg"])
        return {"out": st["out"], "q": st["q"], "k": st["k"], "v": st["v"]}
    if case["mask"] == "llama":
        st["fa"](st["q"], st["k"], st["v"], st["out"], kv_len=st["kv_len"], q_len=st["q_len"],
                 mask_mode=sa.MASK_EXPLICIT, mask=st["mask"])
    else:
        st["fa"](st["q"], st["k"], st["v"], st["out"], kv_len=st["kv_len"], q_len=st["q_len"],
                 page_table=st["table"])
    return st["out"]


# ---- the same in 64 bits ----

def _plain(rows):
    """Cache rows as 64-bit values."""
    if rows.dtype != torch.uint8:
        return rows.double()
    b = rows.reshape(*rows.shape[:-1], -1, 34)
    d = b[..., :2].contiguous().view(torch.float16).double()
    return (d * b[..., 2:].contiguous().view(torch.int8).double()).flatten(-2)


def _q8_query(q):
    """ggml converts the queries of a q8_0 cache to q8_0 blocks first; that is part of what the op computes."""
    b = q.float().reshape(*q.shape[:-1], -1, 32)
    top = b.abs().amax(-1, keepdim=True)
    x = b * torch.where(top > 0, 127.0 / top, torch.zeros_like(top))
    n = torch.sign(x) * torch.floor(x.abs() + 0.5)
    return (n.double() * (top / 127.0).half().double()).reshape(q.shape)


def _stream(cache, table, i, n):
    """Cells 0 .. n-1 of stream i: [n, kv-heads, row]."""
    if table is None:
        return cache[i, :n]
    return cache[table[i, :-(-n // PAGE)].long()].flatten(0, 1)[:n]


def _attention(out, q, k, v, table, cached, rows, exact_new=None):
    d = q.shape[-1]
    for i, (c, r) in enumerate(zip(cached, rows)):
        ks, vs = (_plain(_stream(x, table, i, c + r)) for x in (k, v))
        if exact_new is not None:
            ks[c:], vs[c:] = exact_new[0][i, :r], exact_new[1][i, :r]
        hidden = torch.arange(c + r, device="cuda") > c + torch.arange(r, device="cuda")[:, None]
        for h in range(H):
            g = h // (H // HKV)
            score = q[i, :r, h].contiguous() @ ks[:, g].t().contiguous() / d ** 0.5
            p = torch.softmax(score.masked_fill_(hidden, -math.inf), dim=-1)
            out[i, :r, h] = p @ vs[:, g].contiguous()


def _rope(x, cached):
    """NEOX rotation of the first N_ROT dims at the rows' positions; a row's angles by repeated 32-bit products,
    as the op is specified."""
    pos = (_i32(cached)[:, None] + torch.arange(x.shape[1], device="cuda")).float()
    step = torch.tensor(ROPE_BASE, dtype=torch.float32).pow(-2.0 / N_ROT).cuda()
    angle, angles = pos, []
    for _ in range(N_ROT // 2):
        angles.append(angle)
        angle = angle * step
    a = torch.stack(angles, dim=-1).double()[:, :, None]
    lo, hi = x[..., :N_ROT // 2], x[..., N_ROT // 2:N_ROT]
    return torch.cat([lo * a.cos() - hi * a.sin(), hi * a.cos() + lo * a.sin(), x[..., N_ROT:]], dim=-1)


def _norm(x, weight):
    x = x.double()
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * weight.double()


def exact(case, seed):
    st = _inputs(case, seed)
    cached, rows = _lengths(case)
    if case["kind"] == "gdn":
        return _exact_gdn(st, case, rows)
    q, d = st.get("q"), _dim(case)
    out = torch.zeros((case["streams"], case["rows"], H, d), dtype=torch.float64, device="cuda")
    if case["kind"] == "attend":
        q = _q8_query(q) if case["kv"] == "q8_0" else q.double()
        _attention(out, q, st["k"], st["v"], st["table"], cached, rows)
        return out
    q = _rope(_norm(st["qg"][..., :d], st["q_norm"]), cached)
    k_new, v_new = _rope(_norm(st["k_new"], st["k_norm"]), cached), st["v_new"].double()
    _attention(out, q, st["k"], st["v"], st["table"], cached, rows, (k_new, v_new))
    out *= torch.sigmoid(st["qg"][..., d:].double())
    k, v = st["k"].double(), st["v"].double()
    for i, (c, r) in enumerate(zip(cached, rows)):
        q[i, r:] = 0
        for j in range(r):
            page, cell = int(st["table"][i, (c + j) // PAGE]), (c + j) % PAGE
            k[page, cell], v[page, cell] = k_new[i, j], v_new[i, j]
    return {"out": out, "q": q, "k": k, "v": v}


def _exact_gdn(st, case, rows):
    s = st["state"].double()
    q, k, v, alpha, beta = (st[n].double() for n in ("q", "k", "v", "alpha", "beta"))
    y = torch.zeros_like(v)
    n = _i32(rows)
    snap = n if st["snap"] is None else torch.minimum(st["snap"], n)
    kept = s.clone()
    for j in range(case["rows"]):
        a, b = alpha[:, j, :, None], beta[:, j, :, None]
        read = (s * k[:, j, :, None, :]).sum(-1)
        delta = b * (v[:, j] - (a * read if case["decay_first"] else read))
        s = a[..., None] * s + delta[..., None] * k[:, j, :, None, :]
        live = (n > j)[:, None, None]
        y[:, j] = torch.where(live, (s * q[:, j, :, None, :]).sum(-1), y[:, j])
        kept = torch.where((snap == j + 1)[:, None, None, None], s, kept)
    return {"y": y, "state": kept}


def tolerance(case):
    # about four times what each path shows against 64 bits: 32-bit sums in the recurrence (2e-7 after 16 rows and
    # after 2048; room for another order of the sums), f16 probabilities over queries that were f16 already (1.9e-4),
    # f16 queries, probabilities and partial results elsewhere (4.6e-4; 7.2e-4 with q8_0 blocks rounded to f16)
    if case["kind"] == "gdn":
        return {"rel": 2e-6}
    if case["kind"] == "attend" and case["kv"] == "q8_0":
        return {"rel": 3e-3}
    return {"rel": 8e-4 if _half_q(case) and case["rows"] > 16 else 2e-3}
