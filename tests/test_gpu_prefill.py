"""GPU parity of the chunked-prefill path (blocks of more than 96 rows per GQA group)
against the oracle, through the C ABI.

Bar: max-abs <= 2e-3 and rel-L2 <= 1e-3 on the f32 output against the oracle's
f32-accumulator restatement of ggml's CPU flash_attn_ext.  At full chunk size the oracle
checks row slices: rows [a, b) of a chunk over kv_len cached cells are exactly a block of
b - a rows over kv_len + a cached cells (same cells, same causal rule).
"""
import ctypes
import sys

import numpy as np
import pytest
import torch

import oracle
import sixi_attn as sa
from sixi_attn import workloads as wl

pytestmark = pytest.mark.gpu

MAX_ABS = 2e-3
REL_L2 = 1e-3
# split against unsplit: each side rounds the probabilities to f16 against other exponent references, an
# error of 2^-10 / sqrt(12) / m for significands m, 2.07e-4 rms over log-uniform ones, independent over the
# cells and of the other side's: sqrt(2) times that, 2.93e-4, of the sums (whose f32 order adds 1e-7); a
# third for the spread of few rows
SPLIT_REL_L2 = 3.9e-4


def _say(msg):
    print(f"[gpu-case] {msg}", file=sys.stderr, flush=True)


@pytest.fixture(scope="module")
def fa():
    assert torch.cuda.is_available(), "the gpu tests need a GPU"
    sa.load_library()
    return sa.FlashAttnExt()


def _run(fa, w, dev, mask_mode=sa.MASK_BLOCK_CAUSAL, q=None, mask=None):
    out = torch.full((w.S, w.n_q, w.H, w.D), float("nan"), dtype=torch.float32, device="cuda")
    fa(dev["q"] if q is None else q, dev["k"], dev["v"], out, kv_len=dev["kv_len"], q_len=dev["q_len"],
       mask_mode=mask_mode, mask=mask)
    torch.cuda.synchronize()
    return out.cpu().numpy()


def _check(want, got, label):
    m = oracle.diff_metrics(want, got)
    _say(f"{label} max_abs={m['max_abs']:.3e} rel_l2={m['rel_l2']:.3e}")
    assert np.all(np.isfinite(got))
    assert m["max_abs"] <= MAX_ABS and m["rel_l2"] <= REL_L2, m


def _slice_host(host, s, a, b):
    """rows [a, b) of stream s as a one-stream block with kv_len + a cached cells."""
    kl = int(host["kv_len"][s])
    q = host["q"][s:s + 1, a:b]
    if q.dtype == np.float16:
        q = q.astype(np.float32)
    return {"q": np.ascontiguousarray(q), "k": host["k"][s:s + 1], "v": host["v"][s:s + 1],
            "kv_len": np.array([kl + a], np.int32), "q_len": np.array([b - a], np.int32)}


@pytest.mark.parametrize("name", ["prefill_chunk0", "prefill_chunk1"])
def test_prefill_chunks_parity_every_row(fa, name):
    """All 2048 rows of the chunk against the oracle, on the whole and per 128-row block (the
    prefill kernel's work-group), so a fault in one row block cannot hide in the aggregate."""
    _say(f"config {name} (every row)")
    w = wl.config(name)
    host = wl.make_host(w, poison=True)
    dev = wl.to_device(host)
    got = _run(fa, w, dev)
    want = oracle.attention_for_workload(host, w.kv_type)
    _check(want[0], got[0], f"{name} rows [0,{w.q_len[0]})")
    for a in range(0, w.q_len[0], 128):
        m = oracle.diff_metrics(want[0, a:a + 128], got[0, a:a + 128])
        assert m["max_abs"] <= MAX_ABS and m["rel_l2"] <= REL_L2, (a, m)
    # a row slice is the same block over a longer cache: the slice's oracle agrees
    a, b = 1000, 1100
    sl = oracle.attention_for_workload(_slice_host(host, 0, a, b), w.kv_type)
    _check(sl[0], got[0, a:b], f"{name} rows [{a},{b}) as their own block")


@pytest.mark.parametrize("kv_len,q_len,H,Hkv", [
    ([0, 100, 1000], [130, 257, 17], 24, 4),   # ragged rows, empty cache, a stream under one row block
    ([64, 3], [200, 129], 8, 8),               # no GQA
    ([777, 5], [7, 300], 32, 2),               # 16 q-heads per kv-head
])
def test_ragged_prefill(fa, kv_len, q_len, H, Hkv):
    _say(f"ragged prefill kv_len={kv_len} q_len={q_len} H={H} Hkv={Hkv}")
    w = wl.Workload("ragged_prefill", 0x51A7_3000 + sum(q_len), len(kv_len), kv_len, q_len, H=H, Hkv=Hkv)
    host = wl.make_host(w, poison=True)
    dev = wl.to_device(host)
    got = _run(fa, w, dev)
    want = oracle.attention_for_workload(host, w.kv_type)
    rows_g = np.concatenate([got[s, :q_len[s]].ravel() for s in range(w.S)])
    rows_w = np.concatenate([want[s, :q_len[s]].ravel() for s in range(w.S)])
    _check(rows_w, rows_g, "ragged prefill")


def _small_prefill():
    w = wl.Workload("small_prefill", 0x51A7_4000, 2, [300, 50], [200, 160])
    host = wl.make_host(w, poison=True)
    return w, host, wl.to_device(host)


def test_prefill_mask_none(fa):
    _say("prefill, mask NONE over kv_len + q_len cells")
    w, host, dev = _small_prefill()
    got = _run(fa, w, dev, mask_mode=sa.MASK_NONE)
    want = oracle.attention_for_workload(host, w.kv_type, causal=False)
    for s in range(w.S):
        _check(want[s, :w.q_len[s]], got[s, :w.q_len[s]], f"mask NONE stream {s}")


def test_prefill_explicit_mask_matches_causal(fa):
    _say("prefill, explicit llama mask vs block-causal")
    w, host, dev = _small_prefill()
    a = _run(fa, w, dev)
    n_kv = dev["k"].shape[1]
    mask = torch.from_numpy(oracle.build_kq_mask(n_kv, w.n_q, w.kv_len, w.q_len, True)).view(torch.float16).cuda()
    b = _run(fa, w, dev, mask_mode=sa.MASK_EXPLICIT, mask=mask)
    want = oracle.attention_for_workload(host, w.kv_type)
    for s in range(w.S):
        _check(want[s, :w.q_len[s]], b[s, :w.q_len[s]], f"explicit mask stream {s}")
        assert np.max(np.abs(a[s, :w.q_len[s]] - b[s, :w.q_len[s]])) <= 1e-3


def test_prefill_row_ignores_later_cells_bitwise(fa):
    _say("prefill row j independent of cells > kv_len + j")
    w, host, dev = _small_prefill()
    base = _run(fa, w, dev)
    j = 150
    k2 = dev["k"].clone()
    v2 = dev["v"].clone()
    for s in range(w.S):
        k2[s, w.kv_len[s] + j + 1:] = -3.0
        v2[s, w.kv_len[s] + j + 1:] = 7.0
    alt = _run(fa, w, dict(dev, k=k2, v=v2))
    assert np.array_equal(base[:, :j + 1], alt[:, :j + 1])


def test_prefill_repeatable_bitwise(fa):
    _say("prefill 10 launches, bitwise")
    w, host, dev = _small_prefill()
    first = _run(fa, w, dev)
    for _ in range(9):
        assert np.array_equal(first, _run(fa, w, dev), equal_nan=True)


def test_prefill_f16_queries(fa):
    _say("prefill f16 Q")
    w, host, dev = _small_prefill()
    q16 = dev["q"].to(torch.float16)
    got = _run(fa, w, dev, q=q16)
    ref_host = dict(host)
    ref_host["q"] = q16.float().cpu().numpy()
    want = oracle.attention_for_workload(ref_host, w.kv_type)
    for s in range(w.S):
        _check(want[s, :w.q_len[s]], got[s, :w.q_len[s]], f"f16 Q stream {s}")


def _sizes(fa, p):
    least, full = ctypes.c_size_t(0), ctypes.c_size_t(0)
    assert fa.lib.sixi_attn_workspace_range(ctypes.byref(p), ctypes.byref(least), ctypes.byref(full)) == sa.OK
    assert least.value < full.value, "the case is meant to split"
    return least.value, full.value


def _forward(fa, p, split, ws=None):
    """sixi_attn_forward of `p` with or without the split, on a workspace of its own full of NaN bits."""
    least, full = _sizes(fa, p)
    if split:
        p.flags |= sa.FLAG_SPLIT_PREFILL
    if ws is None:
        ws = torch.full((full if split else least,), 0xFF, dtype=torch.uint8, device="cuda")
    p.stream = torch.cuda.current_stream().cuda_stream
    p.workspace, p.workspace_bytes = ws.data_ptr(), ws.numel()
    rc = fa.lib.sixi_attn_forward(ctypes.byref(p))
    assert rc == sa.OK, sa.strerror(rc)
    torch.cuda.synchronize()


@pytest.mark.parametrize("D", [128, 256])
def test_prefill_writes_no_workspace_unless_asked(fa, D):
    """Without FLAG_SPLIT_PREFILL an f16 prefill leaves the workspace as it is however large it is
    (another call may be using it), and so also runs with one whose unused tail meets a view."""
    _say(f"large workspace, no split D={D}")
    w = wl.Workload("whole prefill", 0x51A7_5300 + D, 1, [3000], [40], D=D)
    host = wl.make_host(w)
    dev = wl.to_device(host)
    out = torch.empty((1, 40, w.H, D), dtype=torch.float32, device="cuda")
    p = fa.params(dev["q"], dev["k"], dev["v"], out, kv_len=dev["kv_len"], q_len=dev["q_len"])
    ws = torch.full((64 << 20,), 0xA5, dtype=torch.uint8, device="cuda")
    _forward(fa, p, False, ws)
    assert bool(torch.all(ws == 0xA5))
    want = oracle.attention_for_workload(host, w.kv_type)
    _check(want, out.cpu().numpy(), "whole")
    # the same queries behind 1 MB of workspace that is declared to run through them
    tail = torch.zeros((1 << 20) + dev["q"].numel() * 4, dtype=torch.uint8, device="cuda")
    q = tail[1 << 20:].view(torch.float32).view(dev["q"].shape)
    q.copy_(dev["q"])
    out2 = torch.empty_like(out)
    _forward(fa, fa.params(q, dev["k"], dev["v"], out2, kv_len=dev["kv_len"], q_len=dev["q_len"]), False, tail)
    assert torch.equal(out, out2)


def _paged(x):
    """A contiguous cache [S, cells, heads, row] as a pool of shuffled 256-cell pages, and its table."""
    S, n = x.shape[0], x.shape[1] // 256
    order = torch.randperm(S * n, generator=torch.Generator().manual_seed(5)).cuda()
    pages = x[:, :n * 256].reshape(S * n, 256, *x.shape[2:])
    pool = torch.empty_like(pages)
    pool[order] = pages
    return pool, order.to(torch.int32).view(S, n)


@pytest.mark.parametrize("kv_len,q_len,H,Hkv,D,kv,mode", [
    ([1500], [17], 24, 4, 128, sa.TYPE_F16, "lengths"),         # 102 rows: one row block, 26 of its rows empty
    ([700, 0, 5], [22, 17, 0], 24, 4, 256, sa.TYPE_F16, "lengths"),  # a second block of 4 rows; one share of one tile
    ([4100], [65], 8, 2, 128, sa.TYPE_Q8_0, "lengths"),         # three blocks, 66 tiles, q8_0
    ([3000, 900], [33, 20], 24, 4, 256, sa.TYPE_Q8_0, "lengths"),
    ([17500], [20], 24, 4, 128, sa.TYPE_F16, "paged"),           # 69 pages: shares that start past the first 64
    ([3000, 900], [33, 20], 24, 4, 256, sa.TYPE_Q8_0, "paged"),
    ([2000, 30], [40, 31], 24, 4, 128, sa.TYPE_F16, "causal"),    # the causal mask, handed over
    ([2000, 30], [40, 31], 24, 4, 256, sa.TYPE_F16, "causal"),
    ([2000, 300], [40, 31], 24, 4, 256, sa.TYPE_F16, "holes"),    # a mask with holes: the staged-mask body
    ([2000, 300], [40, 31], 24, 4, 128, sa.TYPE_Q8_0, "holes"),
    ([1100], [24], 24, 4, 128, sa.TYPE_F16, "softcap"),          # the per-cell body
    ([1100, 600], [24, 20], 24, 4, 256, sa.TYPE_F16, "alibi"),
])
def test_split_row_blocks(fa, kv_len, q_len, H, Hkv, D, kv, mode):
    """Few row blocks over a long cache: several work-groups share the cells of each.  Every stream and head
    against the oracle (the bar above); bit for bit the same when called again; and against the call
    without the split (SPLIT_REL_L2)."""
    _say(f"split kv_len={kv_len} q_len={q_len} H={H} Hkv={Hkv} D={D} kv={kv} {mode}")
    w = wl.Workload("split_prefill", 0x51A7_5100 + sum(q_len) + D, len(kv_len), kv_len, q_len, H=H, Hkv=Hkv, D=D, kv_type=kv)
    host = wl.make_host(w, poison=True)
    dev = wl.to_device(host)
    kw = dict(kv_len=dev["kv_len"], q_len=dev["q_len"])
    k, v, n_kv = dev["k"], dev["v"], dev["k"].shape[1]
    if mode == "paged":
        (k, kw["page_table"]), (v, _) = _paged(k), _paged(v)
    last = np.array(kv_len)[:, None, None] + np.arange(w.n_q)[None, :, None]
    cells = np.arange(n_kv)[None, None]
    seen = (cells <= last) & (np.arange(w.n_q)[None, :, None] < np.array(q_len)[:, None, None])
    if mode == "holes":
        seen &= cells % 7 != 3
    mask = np.where(seen, -0.02 * (last - cells) if mode == "alibi" else 0.0, -np.inf).astype(np.float16)[:, None]
    cap = 20.0 if mode == "softcap" else 0.0
    bias = 8.0 if mode == "alibi" else 0.0
    if mode in ("causal", "holes", "alibi"):
        kw.update(mask_mode=sa.MASK_EXPLICIT, mask=torch.from_numpy(mask).cuda())
    kw.update(logit_softcap=cap, max_bias=bias)
    outs = []
    for split in (True, False, True):
        out = torch.full((w.S, w.n_q, w.H, w.D), float("nan"), dtype=torch.float32, device="cuda")
        _forward(fa, fa.params(dev["q"], k, v, out, **kw), split)
        outs.append(out.cpu().numpy())
    got, whole, again = outs
    assert np.array_equal(got, again, equal_nan=True)
    n = int(max(c + r for c, r in zip(kv_len, q_len)))
    want = oracle.flash_attn_ext(host["q"], np.ascontiguousarray(host["k"][:, :n]), np.ascontiguousarray(host["v"][:, :n]), kv,
                                 np.ascontiguousarray(mask[..., :n]).view(np.uint16), max_bias=bias, logit_softcap=cap)
    for s, r in enumerate(q_len):
        assert np.all(np.isnan(got[s, r:]))  # rows past q_len are not written
        if r == 0:
            continue
        for h in range(H):
            _check(want[s, :r, h], got[s, :r, h], f"stream {s} head {h}")
        m = oracle.diff_metrics(whole[s, :r], got[s, :r])
        _say(f"stream {s}, split against whole: rel_l2={m['rel_l2']:.3e}")
        assert m["rel_l2"] <= SPLIT_REL_L2, m


def test_split_calls_of_two_streams_on_one_handle(fa):
    """One handle, prompts of different streams in turn on two streams that run at once: every output is the
    one its call gives alone."""
    ws = [wl.Workload("two streams", 0x51A7_5600 + i, 1, [n], [r], D=d)
          for i, (n, r, d) in enumerate(((6000, 40, 256), (5000, 64, 128)))]
    devs = [wl.to_device(wl.make_host(w)) for w in ws]

    def call(i):
        out = torch.empty((1, ws[i].n_q, ws[i].H, ws[i].D), dtype=torch.float32, device="cuda")
        d = devs[i]
        fa(d["q"], d["k"], d["v"], out, kv_len=d["kv_len"], q_len=d["q_len"])
        return out

    _say("two streams, one handle")
    alone = [call(i) for i in range(2)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    outs = []
    for _ in range(20):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                outs.append((i, call(i)))
    torch.cuda.synchronize()
    for i, out in outs:
        assert torch.equal(out, alone[i])


@pytest.mark.parametrize("D", [128, 256])
def test_split_row_blocks_at_scale_0(fa, D):
    """A scale of 0 weighs every cell alike: each output is the mean of V, split as unsplit.  One
    stream fills the cache, the other one tile of it, which most of its work-groups see nothing of;
    no mask, so every tile is whole.  Against 64 bits."""
    _say(f"split scale=0 D={D}")
    S, n_q, H, Hkv, n_kv = 2, 22, 24, 4, 4096
    cells = [n_kv, 64]
    gen = torch.Generator(device="cuda").manual_seed(77)
    q = 0.5 * torch.randn((S, n_q, H, D), generator=gen, device="cuda")
    k, v = (torch.randn((S, n_kv, Hkv, D), generator=gen, device="cuda", dtype=torch.float16) for _ in range(2))
    kv_len = torch.tensor([c - n_q for c in cells], dtype=torch.int32, device="cuda")
    out = torch.full((S, n_q, H, D), float("nan"), dtype=torch.float32, device="cuda")
    fa(q, k, v, out, kv_len=kv_len, mask_mode=sa.MASK_NONE, scale=0.0)
    torch.cuda.synchronize()
    got, v = out.cpu().numpy(), v.cpu().double().numpy()
    for s in range(S):
        mean = np.repeat(v[s, :cells[s]].mean(0), H // Hkv, axis=0)
        _check(np.broadcast_to(mean, got[s].shape), got[s], f"stream {s}")


def test_split_in_the_fixed_scratch(fa):
    """sixi_attn_forward_noalloc splits on request with as many shares as its 32 MiB hold: all of a small
    call's, which then equals sixi_attn_forward bit for bit, and seven of the eight that 32 row blocks
    at 256 dims would leave (33.8 MB); without the request it equals the unsplit call."""
    for kv_len, q_len, D, fits in (([3000], [40], 128, True), ([12000, 500, 900, 40], [40, 40, 33, 40], 256, False)):
        _say(f"noalloc split kv_len={kv_len} D={D}")
        w = wl.Workload("noalloc split", 0x51A7_5400 + D, len(kv_len), kv_len, q_len, D=D)
        host = wl.make_host(w, poison=True)
        dev = wl.to_device(host)
        want = oracle.attention_for_workload(host, w.kv_type)
        for split in (True, False):
            outs = []
            for noalloc in (True, False):
                out = torch.full((w.S, w.n_q, w.H, D), float("nan"), dtype=torch.float32, device="cuda")
                p = fa.params(dev["q"], dev["k"], dev["v"], out, kv_len=dev["kv_len"], q_len=dev["q_len"])
                if noalloc:
                    p.flags |= sa.FLAG_SPLIT_PREFILL if split else 0
                    p.stream = torch.cuda.current_stream().cuda_stream
                    assert fa.lib.sixi_attn_forward_noalloc(ctypes.byref(p)) == sa.OK
                    torch.cuda.synchronize()
                else:
                    _forward(fa, p, split)
                outs.append(out.cpu().numpy())
            same = np.array_equal(outs[0], outs[1], equal_nan=True)
            assert same == (fits or not split)
            for s in range(w.S):
                _check(want[s, :q_len[s]], outs[0][s, :q_len[s]], f"stream {s} split={split}")


@pytest.mark.parametrize("D", [128, 256])
@pytest.mark.parametrize("cached", [0, 87, 216, 3000])
@pytest.mark.parametrize("masked", [False, True])
def test_shares_follow_the_cells_in_use(fa, masked, cached, D):
    """A split launch is sized for the cache (16384 cells, NaN past the stream's); the cells in use decide
    how many work-groups share them, at least 128 cells each (40 rows behind 216 cells: two shares), and
    the others write nothing, also where a llama mask's lengths are taken from the mask.  With one share the sums are left alone and the output is the unsplit
    call's bit for bit; always against the oracle."""
    _say(f"short stream in a long cache: cached={cached} D={D} masked={masked}")
    w = wl.Workload("short stream", 0x51A7_5500 + cached + D, 1, [cached], [40], D=D)
    host = wl.make_host(w)
    dev = wl.to_device(host)
    k, v = (torch.full((1, 16384, w.Hkv, D), float("nan"), dtype=torch.float16, device="cuda") for _ in range(2))
    for x, c in ((k, dev["k"]), (v, dev["v"])):
        x[:, :cached + 40] = c.view(torch.float16)[:, :cached + 40]
    mask = None
    if masked:
        mask = torch.from_numpy(wl.kq_mask(16384, 40, w.kv_len, w.q_len)).view(torch.float16).cuda()
    outs = []
    for split in (True, False):
        out = torch.full((1, 40, w.H, D), float("nan"), dtype=torch.float32, device="cuda")
        p = fa.params(dev["q"], k, v, out, kv_len=dev["kv_len"], q_len=dev["q_len"],
                      mask_mode=sa.MASK_EXPLICIT if masked else sa.MASK_BLOCK_CAUSAL, mask=mask)
        least, full = _sizes(fa, p)
        ws = torch.full((full if split else least,), 0xA5, dtype=torch.uint8, device="cuda")
        _forward(fa, p, split, ws)
        outs.append(out.cpu().numpy())
        if split:
            blocks, slot = 4 * 2, 128 * (D + 2) * 4   # kv-heads x row blocks of 40 x 6 rows; bytes of a share
            launched = (full - least) // (blocks * slot)
            sums = ws[least:least + blocks * launched * slot].view(blocks, launched, slot)
            shares = max(1, min(launched, (cached + 40) // 128))
            assert launched > 2 and shares == {0: 1, 87: 1, 216: 2, 3000: launched}[cached]
            assert bool(torch.all(sums[:, shares if shares > 1 else 0:] == 0xA5))
            if shares > 1:
                assert not bool(torch.any(torch.all(sums[:, :shares] == 0xA5, dim=-1)))
    if cached < 216:
        assert np.array_equal(outs[0], outs[1])
    want = oracle.attention_for_workload(host, w.kv_type)
    _check(want, outs[0], "split")
