"""GPU gated-delta-rule verify (sixi_gdn_verify) against the oracle, through the C ABI.

The bar is the reference's own for its GPU step (tests/test_cuda_kernels.cpp:330-339): max-abs
below 1e-4 and cosine above 0.99999 on y and on the state; here also rel-L2 below 1e-5.  Sums over
the state columns run in a different order than the reference's serial loops (partial sums of 16
columns, then a lane tree), so results agree to f32 rounding, not bitwise; repeated launches are
bitwise identical, as the reference's test requires of its kernel.
"""
import sys

import numpy as np
import pytest
import torch

import oracle
import sixi_attn as sa
from test_oracle_gdn import reference_test_inputs

pytestmark = pytest.mark.gpu


def _say(msg):
    print(f"[gpu-case] {msg}", file=sys.stderr, flush=True)


@pytest.fixture(scope="module", autouse=True)
def lib():
    assert torch.cuda.is_available(), "the gpu tests need a GPU"
    return sa.load_library()


def _inputs(S, n, G, K, HD, seed):
    rng = np.random.default_rng(seed)
    k = rng.standard_normal((S, n, G, K))
    k /= np.linalg.norm(k, axis=-1, keepdims=True)                     # unit keys, as after the l2 norm
    q = rng.standard_normal((S, n, G, K)) / np.sqrt(K)
    v = rng.standard_normal((S, n, G, HD))
    al = rng.uniform(0.8, 1.0, (S, n, G))
    be = rng.uniform(0.0, 1.0, (S, n, G))
    S0 = rng.standard_normal((S, G, HD, K)) * 0.5
    return [x.astype(np.float32) for x in (q, k, v, al, be, S0)]


def _check(got, want, label):
    m = oracle.diff_metrics(want, got)
    _say(f"{label}: max_abs={m['max_abs']:.3e} rel_l2={m['rel_l2']:.3e} cos={m['cosine']:.7f}")
    assert np.all(np.isfinite(got)), label
    assert m["max_abs"] < 1e-4 and m["cosine"] > 0.99999 and m["rel_l2"] < 1e-5, (label, m)


def _run(q, k, v, al, be, S0, q_len=None, snap=None, decay_first=False, in_place=True, label=""):
    S, n, G, K = q.shape
    HD = v.shape[-1]
    _say(f"gdn {label}: S={S} n={n} G={G} K={K} HD={HD} q_len={q_len} snap={snap} decay_first={decay_first} "
         f"in_place={in_place}")
    d = [torch.from_numpy(x).cuda() for x in (q, k, v, al, be)]
    st_in = torch.from_numpy(S0).cuda()
    st_out = st_in if in_place else torch.full_like(st_in, float("nan"))
    y = torch.full((S, n, G, HD), float("nan"), dtype=torch.float32, device="cuda")
    ql = torch.tensor(q_len, dtype=torch.int32, device="cuda") if q_len is not None else None
    sn = torch.tensor(snap, dtype=torch.int32, device="cuda") if snap is not None else None
    sa.gdn_verify(*d, y, st_in, None if in_place else st_out, ql, sn, decay_first)
    torch.cuda.synchronize()
    want_y, want_st = oracle.gdn_verify(q, k, v, al, be, S0, q_len, snap, decay_first)
    got_y = y.cpu().numpy()
    assert np.array_equal(np.isnan(got_y), np.isnan(want_y)), f"{label}: rows past q_len written or missing"
    valid = ~np.isnan(want_y)
    _check(got_y[valid], want_y[valid], f"{label} y")
    _check(st_out.cpu().numpy(), want_st, f"{label} state")
    return got_y, st_out.cpu().numpy()


def test_reference_kernel_test_case():
    """tests/test_cuda_kernels.cpp:259-341: 16 groups, state 64, head 128, 8 steps."""
    args = reference_test_inputs()
    y1, s1 = _run(*args, label="reference test case")
    y2, s2 = _run(*args, label="reference test case, again")
    assert np.array_equal(y1, y2) and np.array_equal(s1, s2)        # bitwise repeatable


# 128-dim keys run one of two kernels: up to 64 states of 128 rows (128 of 64) the one whose work-groups
# of 32 state rows fit the 256 CUs at once, beyond that the one with 64 rows per work-group.  (streams,
# groups) on either side of the line:
BOTH_KERNELS = pytest.mark.parametrize("S,G", [(2, 6), (12, 6)])


@pytest.mark.parametrize("decay_first", [False, True])
def test_qwen_verify_block(decay_first):
    # 48 value heads of 128 with 128-dim keys (ssm_time_step_rank 48, ssm_state_size 128), 16 rows
    args = _inputs(6, 16, 48, 128, 128, 11)
    _run(*args, q_len=[16, 16, 9, 1, 0, 16], snap=[16, 3, 9, 0, 0, 15], decay_first=decay_first,
         label="qwen verify")


@pytest.mark.parametrize("K,HD", [(64, 64), (64, 128), (128, 64)])
def test_other_shapes_out_of_place(K, HD):
    args = _inputs(3, 5, 7, K, HD, 20 + K + HD)
    _run(*args, q_len=[5, 2, 4], in_place=False, label=f"K={K} HD={HD}")


@pytest.mark.parametrize("S,G", [(2, 4), (12, 6)])
def test_long_block_several_staging_passes(S, G):
    args = _inputs(S, 40, G, 128, 128, 31)                           # 16 + 16 + 8 rows
    _run(*args, q_len=[40, 33] * (S // 2), snap=[17, 33, 40, 16][:S] * max(1, S // 4), label="40 rows")


@pytest.mark.parametrize("decay_first", [False, True])
@pytest.mark.parametrize("S,G", [(3, 7), (12, 11)])
def test_64_row_states_of_128_dim_keys(S, G, decay_first):
    # 42 work-groups of 32 state rows, and 264: one more than a multiple of 8 states over the line
    n = 40
    q_len = [40, 17, 33, 0, 16, 1, 32, 40, 15, 39, 31, 2][:S]
    snap = [39, 17, 16, 0, 3, 0, 32, 1, 15, 17, 30, 2][:S]
    _run(*_inputs(S, n, G, 128, 64, 91 + S), q_len=q_len, snap=snap, decay_first=decay_first,
         in_place=decay_first, label="64-row states")


@pytest.mark.parametrize("decay_first", [False, True])
def test_several_items_per_work_group(decay_first):
    # 32 streams x 48 groups x 2 halves = 3072 items of 64 state rows: more than the work-groups
    # that fit the device at once (768 on MI355X), so each work-group runs several items and reads
    # the next item's state while it computes the current one; ragged lengths (0, 1, a chunk and a
    # half, every row), snapshot rows anywhere in the block, in place
    S, n, G = 32, 24, 48
    args = _inputs(S, n, G, 128, 128, 71 + int(decay_first))
    rng = np.random.default_rng(72 + int(decay_first))
    q_len = [int(x) for x in rng.integers(0, n + 1, S)]
    q_len[:4] = [0, 1, n, 16]
    snap = [int(rng.integers(0, ql + 1)) for ql in q_len]
    snap[2:4] = [17, 16]
    _run(*args, q_len=q_len, snap=snap, decay_first=decay_first, label="3072 items")


@pytest.mark.parametrize("S,G", [(16, 48), (3, 20)])
def test_strided_views(S, G):
    # ggml views that are not packed: q and k stored group-major ([S][G][n][K] seen as [S][n][G][K]),
    # v, y and both states in padded rows, alpha and beta every other float; out of place, so the
    # padding of y and of the output state must stay untouched; 16 streams x 48 groups = 1536 items
    # (several per work-group, the XCD pairing on), and 60 states in one round of work-groups of 32
    # state rows; blocks of up to 20 rows
    n, K, HD = 20, 128, 128
    q, k, v, al, be, S0 = _inputs(S, n, G, K, HD, 81)
    rng = np.random.default_rng(82)
    q_len = [int(x) for x in rng.integers(0, n + 1, S)]
    q_len[:3] = [n, 0, 16]
    snap = [int(rng.integers(0, ql + 1)) for ql in q_len]
    snap[0] = 17

    def dev(x):
        return torch.from_numpy(np.ascontiguousarray(x)).cuda()

    def group_major(x):
        return dev(x.transpose(0, 2, 1, 3)).permute(0, 2, 1, 3)

    def padded(x, pad, fill=0.0):
        buf = torch.full(x.shape[:-1] + (x.shape[-1] + pad,), fill, dtype=torch.float32, device="cuda")
        buf[..., :x.shape[-1]] = dev(x)
        return buf, buf[..., :x.shape[-1]]

    def every_other(x):
        buf = torch.zeros(x.shape[:-1] + (2 * x.shape[-1],), dtype=torch.float32, device="cuda")
        buf[..., ::2] = dev(x)
        return buf[..., ::2]

    _, vd = padded(v, 4)
    _, st_in = padded(S0, 16)
    y_buf, yd = padded(np.full(v.shape, np.nan, np.float32), 8, float("nan"))
    so_buf, st_out = padded(np.full(S0.shape, np.nan, np.float32), 32, float("nan"))
    _say(f"gdn strided views: S={S} n={n} G={G} q_len={q_len} snap={snap}")
    sa.gdn_verify(group_major(q), group_major(k), vd, every_other(al), every_other(be), yd, st_in, st_out,
                  torch.tensor(q_len, dtype=torch.int32, device="cuda"),
                  torch.tensor(snap, dtype=torch.int32, device="cuda"))
    torch.cuda.synchronize()
    want_y, want_st = oracle.gdn_verify(q, k, v, al, be, S0, q_len, snap)
    got_y = yd.cpu().numpy()
    assert np.array_equal(np.isnan(got_y), np.isnan(want_y)), "rows past q_len written or missing"
    valid = ~np.isnan(want_y)
    _check(got_y[valid], want_y[valid], "strided views y")
    _check(st_out.cpu().numpy(), want_st, "strided views state")
    assert torch.isnan(y_buf[..., HD:]).all() and torch.isnan(so_buf[..., K:]).all(), "padding written"


def test_no_lengths():
    _run(*_inputs(2, 3, 3, 128, 128, 41), label="no lengths")


@BOTH_KERNELS
def test_extreme_gates(S, G):
    # alpha 0 resets the state to the row's write, alpha 1 keeps it; beta 0 writes nothing, beta 1
    # writes the whole correction
    q, k, v, al, be, S0 = _inputs(S, 8, G, 128, 128, 51)
    al[:, ::2] = 0.0
    al[:, 1::4] = 1.0
    be[:, :, ::3] = 0.0
    be[:, :, 1::3] = 1.0
    _run(q, k, v, al, be, S0, q_len=[8, 5] * (S // 2), snap=[8, 4] * (S // 2), label="alpha 0/1, beta 0/1")


@pytest.mark.parametrize("decay_first", [False, True])
@pytest.mark.parametrize("G", [6, 18])   # 24 states, and 72: one kernel each
def test_decays_that_leave_the_carried_scale_range(G, decay_first):
    # the kernel carries the state as a scalar times a matrix and folds the scalar in when the
    # running product of the gates leaves [2^-30, 2^30]: gates of 2^-20 (the product leaves the range
    # at the second), 2^-40 (at once), 0 (a reset) and 4 (growth, the product passes 2^30 at the
    # 16th row), across staging passes, against the oracle's step by step recurrence
    q, k, v, al, be, S0 = _inputs(4, 40, G, 128, 128, 61)
    al[0, 3:6] = 2.0 ** -20
    al[1, 10] = 2.0 ** -40
    al[1, 20] = 0.0
    al[2, :] = 4.0
    al[3, 14:18] = 2.0 ** -20
    S, n, _, K = q.shape
    d = [torch.from_numpy(x).cuda() for x in (q, k, v, al, be)]
    st = torch.from_numpy(S0).cuda()
    y = torch.full((S, n, G, 128), float("nan"), dtype=torch.float32, device="cuda")
    snap = [40, 4, 17, 16]
    _say(f"gdn gate range: S={S} n={n} G={G} decay_first={decay_first} snap={snap}")
    sa.gdn_verify(*d, y, st, None, None, torch.tensor(snap, dtype=torch.int32, device="cuda"), decay_first)
    torch.cuda.synchronize()
    want_y, want_st = oracle.gdn_verify(q, k, v, al, be, S0, None, snap, decay_first)
    # the gates of 4 grow the state by up to 4^40: the bar is relative to each stream's scale
    for s in range(S):
        for got, want, what in ((y.cpu().numpy()[s], want_y[s], "y"), (st.cpu().numpy()[s], want_st[s], "state")):
            assert np.all(np.isfinite(got)), (s, what)
            m = oracle.diff_metrics(want, got)
            scale = float(np.abs(want).max())
            _say(f"stream {s} {what}: max_abs/scale={m['max_abs'] / scale:.3e} rel_l2={m['rel_l2']:.3e}")
            assert m["max_abs"] <= 1e-5 * scale and m["rel_l2"] < 1e-5 and m["cosine"] > 0.99999, (s, what, m)


@pytest.mark.parametrize("HD,decay_first", [(128, True), (128, False), (64, True)])
@pytest.mark.parametrize("n,q_len,snap", [
    (1, None, None),                                    # one row
    (15, [15, 1, 0, 7], [0, 1, 0, 7]),                    # under a chunk; no rows; the input state kept
    (17, [17, 16, 17, 3], [16, 16, 17, 2]),               # snapshot at a chunk's last row, a chunk and a row
    (49, [49, 48, 33, 32], [20, 48, 32, 31]),             # three chunks and a row, two to the edge
    (230, [230, 100, 17, 81], [113, 100, 1, 80]),         # every ring slot several times
])
def test_pipelined_chunks_of_few_streams(n, q_len, snap, HD, decay_first):
    """Blocks whose work-groups (32 state rows each) fit the CUs at once: 4 streams x 9 groups, not a
    multiple of 8 states, and (with one row) 8 streams x 4 groups, which are dealt by XCD.  The
    oracle's serial recurrence and the kernel's f32 sums differ by rounding that grows no faster than
    the rows: 230 rows stay within the bar of the 16-row block."""
    args = _inputs(4 if q_len else 8, n, 9 if q_len else 4, 128, HD, 500 + n + HD)
    first = _run(*args, q_len=q_len, snap=snap, decay_first=decay_first, in_place=n % 2 == 0, label=f"{n} rows pipelined")
    again = _run(*args, q_len=q_len, snap=snap, decay_first=decay_first, in_place=n % 2 == 0, label="again")
    assert np.array_equal(first[0], again[0], equal_nan=True) and np.array_equal(first[1], again[1])
