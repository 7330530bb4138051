"""FlashAttnExt's choice of workspaces on the host: the library sizes and validates the calls, a stand-in
takes the launch, so that nothing here touches a device."""
import ctypes
import threading

import pytest
import torch

import sixi_attn as sa

STREAM = 0x5000


class _Library:
    """The library with sixi_attn_forward replaced by `launch(params)`."""

    def __init__(self, launch):
        self._lib, self._launch = sa.load_library(), launch
        self.calls = []

    def __getattr__(self, name):
        fn = getattr(self._lib, name)
        if name == "sixi_attn_forward":
            def fn(ref):
                self._launch(ref._obj)
                return sa.OK

        def call(*args):
            self.calls.append(name)
            return fn(*args)

        return call


@pytest.fixture
def handle(monkeypatch):
    state = {"capturing": False, "launch": lambda p: None}

    class Stream:
        cuda_stream = STREAM

    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: Stream)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state["capturing"])
    fa = sa.FlashAttnExt(device="cpu")
    fa.lib = _Library(lambda p: state["launch"](p))
    return fa, state


def _call(fa, rows=40, n_kv=4096, D=128, q8=False, **kw):
    q = torch.zeros((1, rows, 24, D))
    k = torch.zeros((1, n_kv, 4, D // 32 * 34), dtype=torch.uint8) if q8 else torch.zeros((1, n_kv, 4, D), dtype=torch.float16)
    return fa(q, k, torch.zeros_like(k), torch.zeros((1, rows, 24, D)), kv_len=torch.zeros(1, dtype=torch.int32), **kw)


def _held(fa):
    """Bytes of the tensors the handle keeps."""
    def walk(x):
        if isinstance(x, torch.Tensor):
            return x.numel() * x.element_size()
        if isinstance(x, dict):
            x = list(x.values())
        return sum(map(walk, x)) if isinstance(x, (list, tuple)) else 0

    return walk(vars(fa))


def test_split_calls_of_two_threads_have_a_workspace_each(handle):
    """Two threads on one stream may queue the kernels of two prefill calls in any order: the first one's
    sums must not lie where the second one's will."""
    fa, state = handle
    _call(fa)
    both = threading.Barrier(2, timeout=60)
    ranges = []

    def launch(p):
        assert p.flags & sa.FLAG_SPLIT_PREFILL
        ranges.append((p.workspace, p.workspace + p.workspace_bytes))
        both.wait()  # both calls hold their workspace here

    state["launch"] = launch
    threads = [threading.Thread(target=_call, args=(fa,)) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    (a0, a1), (b0, b1) = ranges
    assert a1 <= b0 or b1 <= a0


def test_split_workspaces_are_given_back(handle):
    fa, _ = handle
    for stream_rows in (17, 40, 64, 100):
        _call(fa, rows=stream_rows)
    assert _held(fa) <= 4096


@pytest.mark.parametrize("q8", [False, True])
def test_an_eager_split_call_sizes_what_the_captured_one_uses(handle, q8, monkeypatch):
    """A captured call must allocate nothing: the eager call before it (which splits, and so runs on
    another buffer) has sized the handle's workspace for it, a q8_0 cache's staging included."""
    fa, state = handle
    _call(fa, q8=q8)
    kept = fa._ws
    used = []
    state.update(capturing=True, launch=lambda p: used.append((p.workspace, p.workspace_bytes, p.flags)))
    monkeypatch.setattr(torch, "empty", lambda *a, **kw: pytest.fail("allocation under capture"))
    _call(fa, q8=q8)
    assert fa._ws is kept
    assert used == [(kept.data_ptr(), kept.numel(), 0)]


def test_who_splits(handle):
    """By default only eager calls on the current stream split; with split_prefill=True the others do, on
    memory that is theirs: the caller's workspace, or (under torch's capture) its pool's."""
    fa, state = handle
    flags = []
    state["launch"] = lambda p: flags.append(bool(p.flags & sa.FLAG_SPLIT_PREFILL))
    ws = torch.empty(128 << 20, dtype=torch.uint8)
    assert ws.data_ptr() % 64 == 0
    for capturing in (False, True):
        state["capturing"] = capturing
        for split in (None, True, False):
            _call(fa, split_prefill=split)
            _call(fa, split_prefill=split, stream=STREAM)  # the current stream, by its handle
            _call(fa, split_prefill=split, stream=STREAM + 8, workspace=ws)
    assert flags == [True, False, False, True, True, True] + [False] * 3 + [False] * 3 + [True] * 3 + [False] * 3
    with pytest.raises(ValueError):
        _call(fa, split_prefill=True, stream=STREAM + 8)


def test_views_hold_what_they_are_given():
    """The packed view against the fields one by one: Python and numpy integers, a null pointer, the
    extents and strides of permuted and sliced tensors."""
    import numpy as np

    for ptr, ne, nb in ((0x7F12_3456_7890, [1, 2, 3, 4], [4, 8, 16, 32]),
                        (None, np.array([1 << 40, 5, 0, -1]), [np.int32(2), -16, 1 << 62, 0])):
        v = sa.make_view(ptr, sa.TYPE_F16, ne, nb)
        assert v.data == ptr and v.type == sa.TYPE_F16 and v.reserved == 0
        assert list(v.ne) == [int(x) for x in ne] and list(v.nb) == [int(x) for x in nb]
    t = torch.zeros((3, 5, 7, 64), dtype=torch.float16).permute(0, 2, 1, 3)[:, 1:, ::2]
    v = sa.view_of(t)
    assert v.data == t.data_ptr() and list(v.ne) == [64, 6, 3, 3]
    assert list(v.nb) == [2, 64 * 2, 2 * 7 * 64 * 2, 5 * 7 * 64 * 2]
    v = sa.view_of(t, tokens_heads=False)
    assert list(v.ne) == [64, 3, 6, 3] and list(v.nb) == [2, 2 * 7 * 64 * 2, 64 * 2, 5 * 7 * 64 * 2]
