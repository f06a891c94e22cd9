"""The 32-bit matrix-core kernels (na_wave.hip: float32, and strided
bf16 / fp16): their window rules against the oracle's windows on the CPU, and
on an MI355X forward + LSE + backward against the float64 oracle at the edges
of their tiles, and non-finite values against the vector-ALU kernels."""

import pytest
import torch

from _helpers import DEV, assert_close, randn
from oracle import na as O
from oracle import window as W


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("K,s", [(1, 1), (3, 1), (3, 2), (3, 3), (5, 2), (5, 4), (7, 3), (7, 7)])
def test_strided_inverse_windows(K, s, causal):
    """A key's queries: of the positions [j <= K-1 ? 0 : j - K/2, j >= L-K ?
    L : j + K/2 + 1) (causal [j, j + K)) every s-th; both ends are
    non-decreasing in j, so a tile of keys has a box of queries no longer
    than (T - 1 + K - 1) / s + 1, or the K - 1 more of a clamped edge."""
    for L in list(range(max(K, 1), 3 * K + 6)) + [40]:
        n_out = -(-L // s)
        idx, valid = W.axis_indices(range(0, L, s), L, K, 1, causal)
        held = [set() for _ in range(L)]
        for o in range(n_out):
            for j, ok in zip(idx[o].tolist(), valid[o].tolist()):
                if ok:
                    held[j].add(o)
        last = (0, 0)
        for j in range(L):
            lo = j if causal else (0 if j <= K - 1 else j - K // 2)
            hi = min(j + K, L) if causal else (L if j >= L - K else j + K // 2 + 1)
            lo, hi = -(-lo // s), min(-(-hi // s), n_out)
            assert set(range(lo, hi)) == held[j], (L, K, s, j)
            assert lo >= last[0] and hi >= last[1]
            last = (lo, hi)


def _ids(cases):
    return [f"{c[0]}-{'x'.join(map(str, c[2]))}-d{c[5]}-k{'x'.join(map(str, c[6]))}"
            f"-s{'x'.join(map(str, c[8]))}" for c in cases]


F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16
# (dtype, B, spatial, H, Hkv, D, kernel, dilation, stride, causal)
CASES = [
    (F32, 1, (1,), 1, 1, 16, (1,), (1,), (1,), (True,)),            # one row
    (F32, 2, (16,), 2, 1, 32, (3,), (1,), (1,), (False,)),          # one whole tile
    (F32, 1, (17,), 3, 3, 64, (15,), (1,), (1,), (False,)),         # one row over
    (F32, 1, (150,), 4, 2, 128, (63,), (2,), (1,), (False,)),       # wide box, phases
    (F32, 2, (13, 11), 2, 2, 32, (7, 7), (1, 1), (1, 1), (False, False)),
    (F32, 1, (9, 33), 2, 1, 16, (3, 5), (3, 2), (1, 1), (False, True)),
    (F32, 1, (14, 17), 6, 2, 64, (5, 7), (1, 1), (2, 3), (False, True)),
    (F32, 1, (6, 9, 10), 2, 1, 32, (3, 5, 3), (1, 1, 3), (1, 2, 1), (True, False, False)),
    (BF16, 2, (31,), 2, 2, 64, (5,), (1,), (4,), (False,)),
    (BF16, 1, (19, 23), 4, 2, 32, (7, 3), (1, 2), (5, 1), (False, False)),
    (F16, 1, (15, 12), 2, 1, 128, (3, 5), (1, 1), (3, 2), (False, False)),
    (F16, 1, (7, 8, 9), 2, 2, 32, (3, 3, 5), (1, 1, 1), (3, 1, 2), (False, True, False)),
]


def _form(which, case):
    from natten_amd._core import hip

    dtype, B, sp, H, Hkv, D, ks, dil, st, caus = case
    q = torch.empty((B, *sp, H, D), dtype=dtype, device="meta")
    k = torch.empty((B, *sp, Hkv, D), dtype=dtype, device="meta")
    return hip.matrix_form(which, q, k, ks, st, dil, caus, 0.3)


@pytest.mark.parametrize("case", CASES, ids=_ids(CASES))
def test_backward_runs_on_matrix_cores(case):
    from natten_amd._core import hip

    assert _form("bwd", case)
    with hip.generic_kernels():
        assert not _form("bwd", case) and not _form("fwd", case)


# Just outside a limit of the float32 matrix-core kernels.
OUTSIDE = [
    (F32, 1, (150,), 1, 1, 48, (7,), (1,), (1,), (False,)),            # head_dim
    (F32, 1, (150,), 1, 1, 32, (8,), (1,), (1,), (False,)),            # even window
    (F32, 1, (150,), 1, 1, 32, (7,), (2,), (3,), (False,)),            # stride and dilation
    (F32, 1, (13, 20), 1, 1, 32, (7, 7), (2, 2), (1, 1), (False, False)),  # d K > L
    (BF16, 1, (31,), 2, 2, 16, (5,), (1,), (2,), (False,)),            # 16 bits, head_dim 16
    (F32, 1, (1 << 20,), 8, 8, 64, (7,), (1,), (1,), (False,)),        # 2^31 bytes a sample
]


# Ragged phases: three points of a tile's 16 rows each.  Both grids of a backward
# hold 64 threads per tile; below and above 2^32 of them.
@pytest.mark.parametrize("B,runs", [(4, True), (5, False)])
def test_launches_stay_below_2_32_threads(B, runs):
    L, d = 24_000_000, 8_000_000
    assert (2 * B * d * 64 < 1 << 32) == runs
    case = (F32, B, (L,), 1, 1, 16, (3,), (d,), (1,), (False,))
    for which in ("bwd", "qk_bwd", "av_bwd"):
        assert _form(which, case) == runs


def test_causal_dilation_past_the_extent():
    """A causal axis of d > L has d phases, most of them empty (the C interface
    takes it): run while the launch holds them, and no overflow past that."""
    for d, runs in ((1000, True), (1 << 20, True), (1 << 25, False), ((1 << 31) - 1, False)):
        case = (F32, 1, (50,), 1, 1, 32, (7,), (d,), (1,), (True,))
        for which in ("fwd", "bwd", "qk", "qk_bwd"):
            assert _form(which, case) == runs, (d, which)


@pytest.mark.parametrize("case", OUTSIDE, ids=_ids(OUTSIDE))
def test_outside_the_limits(case):
    for which in ("fwd", "bwd"):
        assert not _form(which, case)
    if case[8] == (1,) * len(case[8]):
        for which in ("qk", "av", "qk_bwd", "av_bwd"):
            assert not _form(which, case)


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=_ids(CASES))
def test_against_oracle(case):
    import natten_amd

    dtype, B, sp, H, Hkv, D, ks, dil, st, caus = case
    print(f"[case] wave {case}", flush=True)
    fn = {1: natten_amd.na1d, 2: natten_amd.na2d, 3: natten_amd.na3d}[len(sp)]
    q, k, v = (randn((B, *sp, h, D), dtype, i) for i, h in enumerate((H, Hkv, Hkv)))
    ts = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]
    out, lse = fn(*ts, ks, st, dil, caus, return_lse=True)

    def f(a, b, c):
        return O.na_functional(a, b, c, ks, st, dil, caus, return_lse=True)

    ro, rl = f(q, k, v)
    assert_close(out, ro, dtype, "out")
    assert_close(lse, rl, dtype, "lse")
    go, gl = randn(out.shape, dtype, 7), randn(lse.shape, dtype, 8)
    torch.autograd.backward((out, lse), (go.to(DEV), gl.to(DEV)))
    for t, r, n in zip(ts, O.grads(f, (q, k, v), (go, gl)), ("dq", "dk", "dv")):
        assert_close(t.grad, r, dtype, n)


# Forwards that the size decides: (case, runs on matrix cores).
SIZES = [
    ((F32, 2, (500,), 4, 4, 128, (3,), (1,), (1,), (False,)), False),   # one chain per wave
    ((F32, 4, (6000,), 12, 12, 128, (3,), (1,), (1,), (False,)), True),
    ((F32, 2, (500,), 4, 4, 64, (3,), (1,), (1,), (False,)), True),
    ((F32, 1, (67, 42), 4, 4, 64, (3, 3), (1, 1), (3, 3), (False, False)), False),  # 16 boxes
    ((F32, 1, (100, 100), 4, 4, 64, (3, 3), (1, 1), (2, 2), (False, False)), False),
    ((F32, 8, (200, 200), 8, 8, 64, (3, 3), (1, 1), (2, 2), (False, False)), True),
    ((BF16, 1, (59, 90), 4, 4, 128, (3, 3), (1, 1), (2, 2), (False, False)), False),
    ((BF16, 4, (57, 75), 4, 4, 64, (7, 7), (1, 1), (2, 2), (False, False)), True),
    ((F32, 2, (61, 45), 8, 8, 32, (7, 7), (1, 1), (1, 1), (False, False)), True),
]


@pytest.mark.parametrize("case,runs", SIZES, ids=_ids([c for c, _ in SIZES]))
def test_forward_by_size(case, runs):
    from natten_amd._core import hip

    assert _form("fwd", case) == runs
    with hip.any_size_kernels():
        assert _form("fwd", case)


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=_ids(CASES))
def test_forward_at_any_size(case):
    """The forward of every case on matrix cores, also where its size would
    choose the vector ALU."""
    import natten_amd
    from natten_amd._core import hip

    dtype, B, sp, H, Hkv, D, ks, dil, st, caus = case
    print(f"[case] wave forward {case}", flush=True)
    q, k, v = (randn((B, *sp, h, D), dtype, i) for i, h in enumerate((H, Hkv, Hkv)))
    with hip.any_size_kernels():
        assert _form("fwd", case)
        out, lse = hip.fused_forward(q.to(DEV), k.to(DEV), v.to(DEV), ks, st, dil, caus, 0.3)
    ro, rl = O.na_functional(q, k, v, ks, st, dil, caus, 0.3, return_lse=True)
    assert_close(out, ro, dtype, "out")
    assert_close(lse, rl, F32, "lse", scale_tol=1.0 if dtype == F32 else 4.0)


@pytest.mark.gpu
@pytest.mark.parametrize("where", ["q", "k", "v", "grad"])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")], ids=str)
def test_non_finite_values_stay_in_their_windows(where, bad):
    """A tile's product runs over a box wider than its queries' windows; a
    NaN or infinity may reach no more than the vector-ALU kernels let it reach
    (they also give NaN where a window's first score is -inf)."""
    import natten_amd
    from natten_amd._core import hip

    for dtype, st in ((F32, 1), (BF16, 2)):
        ts = [randn((1, 21, 19, 2, 32), dtype, i).to(DEV) for i in range(3)]
        go = randn((1, -(-21 // st), -(-19 // st), 2, 32), dtype, 3).to(DEV)
        bad_t = dict(zip(("q", "k", "v", "grad"), (*ts, go)))[where]
        bad_t[0, 6, 4, 1, 3] = bad
        ts = [t.requires_grad_(True) for t in ts]
        res = []
        for generic in (False, True):
            with hip.generic_kernels(generic):
                out = natten_amd.na2d(*ts, (7, 5), st)
                res.append([out, *torch.autograd.grad(out, ts, go)])
        for a, b in zip(*res):
            fin = torch.isfinite(b)
            assert bool(fin.any()) and bool(torch.isfinite(a[fin]).all())
            assert_close(a[fin], b[fin].double(), dtype, where)
        assert where == "grad" or not bool(torch.isfinite(res[0][0]).all())


# (B, spatial, H, Hkv, D, kernel, dilation, causal): the float32 split ops
SPLIT = [
    (1, (15,), 1, 1, 16, (13,), (1,), (False,)),               # a tile less one row
    (2, (49,), 2, 1, 64, (7,), (3,), (False,)),                # phases, one row over
    (1, (33,), 1, 1, 128, (31,), (1,), (True,)),               # causal: slots before the sample
    (1, (9, 17), 2, 2, 32, (5, 5), (1, 3), (False, False)),
    (2, (8, 13), 4, 2, 16, (3, 7), (2, 1), (True, False)),
    (1, (5, 6, 9), 3, 1, 32, (3, 3, 5), (1, 2, 1), (False, True, False)),
    (1, (24, 24), 1, 1, 32, (21, 23), (1, 1), (False, False)),  # most slots: one wave per group
    (1, (60,), 2, 1, 128, (51,), (1,), (True,)),               # AV of a wide head
]

# Split and position-bias forwards by size: (spatial, B, H, D, kernel) and what runs
# on matrix cores of QK, AV, and of the logits and AV with position bias.
FWD = [
    (((500,), 2, 4, 128, 3), (False, False, False, False)),
    (((6000,), 4, 10, 128, 3), (True, False, False, False)),
    (((500,), 2, 4, 64, 5), (False, False, False, False)),
    (((6000,), 4, 10, 32, 7), (True, False, False, False)),
    (((600,), 2, 5, 128, 9), (True, False, True, False)),
    (((6000,), 6, 12, 32, 9), (True, False, True, True)),
    (((500,), 2, 5, 64, 13), (True, False, True, True)),
    (((500,), 2, 4, 64, 13), (True, False, False, False)),  # few heads, one axis
    (((500,), 2, 4, 64, 31), (True, True, True, True)),
    (((6000,), 4, 10, 64, 13), (True, True, True, True)),
    (((40, 40), 4, 5, 32, 3), (True, False, False, False)),
    (((24, 24), 2, 4, 32, 3), (True, False, True, False)),
    (((40, 40), 4, 5, 16, 5), (True, True, True, True)),
    (((14, 14), 1, 2, 128, 5), (True, False, True, True)),
    (((56, 56), 4, 2, 32, 7), (True, True, True, True)),
]


@pytest.mark.parametrize("problem,want", FWD, ids=[f"{c}" for c, _ in FWD])
def test_split_forwards_by_size(problem, want):
    from natten_amd._core import _lib

    sp, B, H, D, K = problem
    one = (1,) * len(sp)
    case = (F32, B, sp, H, H, D, (K,) * len(sp), one, one, (False,) * len(sp))
    p = _rpb_plan(B, sp, H, D, K, 1, _lib.NA_F32)
    assert (_form("qk", case), _form("av", case), p["qk"] == _lib.RPB_TILE,
            p["av"] == _lib.RPB_TILE) == want


@pytest.mark.parametrize("case", SPLIT, ids=[f"{'x'.join(map(str, c[1]))}-d{c[4]}" for c in SPLIT])
def test_split_backward_runs_on_matrix_cores(case):
    B, sp, H, Hkv, D, ks, dil, caus = case
    for which in ("qk_bwd", "av_bwd"):
        assert _form(which, (F32, B, sp, H, Hkv, D, ks, dil, (1,) * len(sp), caus))
        assert not _form(which, (BF16, B, sp, H, Hkv, D, ks, dil, (1,) * len(sp), caus))


@pytest.mark.gpu
@pytest.mark.parametrize("case", SPLIT, ids=[f"{'x'.join(map(str, c[1]))}-d{c[4]}" for c in SPLIT])
def test_split_against_oracle(case):
    import natten_amd
    from natten_amd import functional as F

    B, sp, H, Hkv, D, ks, dil, caus = case
    print(f"[case] wave split {case}", flush=True)
    r = len(sp)
    qk, av = getattr(F, f"na{r}d_qk"), getattr(F, f"na{r}d_av")
    q, k, v = (randn((B, *sp, h, D), F32, i) for i, h in enumerate((H, Hkv, Hkv)))
    ts = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]
    logits = qk(ts[0], ts[1], ks, dil, is_causal=caus, scale=0.3)
    ref_l = O.na_qk(q, k, ks, 1, dil, caus, 0.3)
    assert_close(logits, ref_l, F32, "logits")
    attn = torch.softmax(ref_l, -1).float()
    ta = attn.to(DEV).requires_grad_(True)
    out = av(ta, ts[2], ks, dil, is_causal=caus)
    assert_close(out, O.na_av(attn, v, ks, 1, dil, caus), F32, "out")
    gl = randn(logits.shape, F32, 7)
    go = randn(out.shape, F32, 8)
    got = (*torch.autograd.grad(logits, ts[:2], gl.to(DEV)),
           *torch.autograd.grad(out, (ta, ts[2]), go.to(DEV)))
    gl = torch.where(torch.isfinite(ref_l), gl.double(), 0.0)  # no gradient at -inf
    ref = (*O.grads(lambda a, b: torch.where(torch.isfinite(ref_l),
                                             O.na_qk(a, b, ks, 1, dil, caus, 0.3), 0.0),
                    (q, k), (gl,)),
           *O.grads(lambda a, b: O.na_av(a, b, ks, 1, dil, caus), (attn, v), (go,)))
    for g, w, n in zip(got, ref, ("dq", "dk", "dattn", "dv")):
        # sums of up to 483 products of unit normals in float32
        assert_close(g, w, F32, n, scale_tol=4.0)


@pytest.mark.gpu
def test_split_non_finite_values_stay_in_their_windows():
    """As above for the AV forward, whose product runs over a box."""
    from natten_amd import functional as F

    q, v, k = (randn((1, 21, 19, 2, 32), F32, i).to(DEV) for i in range(3))
    clean = [F.na2d_av(torch.softmax(F.na2d_qk(q, k, 7), -1), v, 7)]
    v2 = v.clone()
    v2[0, 6, 4, 1, 3] = float("nan")
    out = F.na2d_av(torch.softmax(F.na2d_qk(q, k, 7), -1), v2, 7)
    bad = torch.isnan(out)
    holds = torch.zeros(21, 19, dtype=torch.bool)
    for i in range(21):
        for j in range(19):
            a, b = min(max(i - 3, 0), 14), min(max(j - 3, 0), 12)
            holds[i, j] = a <= 6 < a + 7 and b <= 4 < b + 7
    want = torch.zeros_like(bad)
    want[0, :, :, 1, 3] = holds.to(DEV)
    assert torch.equal(bad, want)
    assert torch.allclose(out[~bad], clean[0][~bad], atol=1e-6)


def _slots(sp, ks, dil, caus):
    """Per query and slot (row-major): the key's token, and whether it counts."""
    tok = torch.zeros((1, 1), dtype=torch.int64)
    good = torch.ones((1, 1), dtype=torch.bool)
    for n, K, d, c in zip(sp, ks, dil, caus):
        idx, ok = (torch.as_tensor(x) for x in W.axis_indices(range(n), n, K, d, c))
        tok = (tok[:, None, :, None] * n + idx[None, :, None, :]).reshape(tok.shape[0] * n, -1)
        good = (good[:, None, :, None] & ok[None, :, None, :]).reshape(tok.shape)
    return tok, good


# (spatial, H, Hkv, D, kernel, dilation, causal, token that holds the bad value)
NONFINITE = [
    ((21, 19), 4, 2, 32, (7, 5), (1, 1), (False, False), 6 * 19 + 4),
    ((17, 22), 2, 1, 64, (5, 3), (2, 3), (True, False), 9 * 22 + 1),
    ((70,), 3, 3, 16, (13,), (3,), (True,), 40),
    ((6, 7, 8), 2, 2, 32, (3, 3, 5), (1, 2, 1), (False, True, False), 150),
]


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [float("nan"), float("inf")], ids=str)
@pytest.mark.parametrize("where", ["q", "k", "v", "attn", "grad"])
@pytest.mark.parametrize("case", NONFINITE, ids=[f"{'x'.join(map(str, c[0]))}" for c in NONFINITE])
def test_split_gradients_keep_non_finite_values_in_their_windows(case, where, bad):
    """Both passes of both backward calls (and so the blocks that compute a
    wave's rows again one by one): non-finite exactly where the window of the bad
    row's query, or the windows that hold the bad row's key, put it."""
    from natten_amd._core import hip

    sp, H, Hkv, D, ks, dil, caus, t = case
    print(f"[case] non-finite split gradients {case} {where} {bad}", flush=True)
    tok, good = _slots(sp, ks, dil, caus)
    n, kk, rep, one = tok.shape[0], tok.shape[1], H // Hkv, (1,) * len(sp)
    h, e, slot = 1, 3, int(good[t].nonzero()[-1])
    q, g = (randn((1, *sp, H, D), F32, i).to(DEV) for i in (0, 1))
    k, v = (randn((1, *sp, Hkv, D), F32, i).to(DEV) for i in (2, 3))
    a, dl = (randn((1, *sp, H, kk), F32, i).to(DEV) for i in (4, 5))

    def run():
        return (*hip.qk_backward(q, k, dl, ks, one, dil, caus, 0.3),
                *hip.av_backward(a, v, g, ks, one, dil, caus))

    clean = run()
    hk = h // rep if where not in ("k", "v") else h % Hkv
    x, head, last = {"q": (q, h, e), "k": (k, hk, e), "v": (v, hk, e), "grad": (g, h, e),
                     "attn": (a, h, slot)}[where]
    x.reshape(n, x.shape[-2], -1)[t, head, last] = bad
    if where == "attn":  # the same slot of the logits' gradient
        dl.reshape(n, H, kk)[t, h, slot] = bad
    want = [torch.zeros((n, *y.shape[-2:]), dtype=torch.bool) for y in clean]
    dq, dk, da, dv = want
    if where == "q":
        dk[tok[t, good[t]], hk, e] = True
    if where == "grad":
        dv[tok[t, good[t]], hk, e] = True
        da[t, h, good[t]] = True
    if where == "attn":
        dq[t, h, :] = True
        dk[tok[t, slot], hk, :] = True
        dv[tok[t, slot], hk, :] = True
    if where in ("k", "v"):
        holds = (tok == t) & good
        for r in range(hk * rep, (hk + 1) * rep):
            if where == "k":
                dq[holds.any(1), r, e] = True
            else:
                da[:, r] |= holds
    for y, c, w, name in zip(run(), clean, want, ("dq", "dk", "dattn", "dv")):
        y, c = (z.reshape(n, *z.shape[-2:]).cpu() for z in (y, c))
        assert torch.equal(~torch.isfinite(y), w), name
        assert_close(y[~w], c[~w].double(), F32, name, scale_tol=4.0)


# (B, spatial, H, D, K, dilation) of the bias partials the dq pass writes;
# empty tiles: short phases with no query in their last tile
BIAS = [
    (2, (97,), 3, 32, 7, 3),       # rank 1: a pass of its own
    (1, (7, 9), 1, 16, 7, 1),      # every window but a few clamped, ragged tiles
    (2, (17, 18), 2, 32, 3, 2),    # empty tiles, phases of two lengths
    (1, (19, 33), 2, 64, 5, 3),
    (3, (24, 40), 2, 32, 7, 1),    # inner tiles (no window clamped) and edges
]


def _rpb_plan(B, sp, H, D, K, d, dtype):
    import ctypes

    from natten_amd._core import _lib

    p = _lib.make_rpb_params(len(sp), B, H, D, sp, (K,) * len(sp), (d,) * len(sp), False, dtype, 0.3)
    plan = _lib.NaRpbPlan()
    assert _lib.load().na_rpb_kernel_plan(ctypes.byref(p), ctypes.byref(plan)) == 0
    return {f: getattr(plan, f) for f, _ in plan._fields_}


@pytest.mark.parametrize("case", BIAS, ids=[f"{'x'.join(map(str, c[1]))}-k{c[4]}d{c[5]}" for c in BIAS])
def test_bias_plans_name_the_kernels(case):
    from natten_amd._core import _lib

    p = _rpb_plan(*case, _lib.NA_F32)
    assert [p[f] for f in ("dq", "dk", "dattn", "dv")] == [_lib.RPB_TILE] * 4
    assert p["fused_bias"] == (len(case[1]) == 2)  # rank 1: a pass of its own
    assert not any(_rpb_plan(*case, _lib.NA_BF16)[f] for f in ("qk", "av", "dq", "dk", "fused_bias"))
    B, sp, H, D, K, d = case
    assert not any(_rpb_plan(B, sp, H, 24, K, d, _lib.NA_F32)[f] for f in ("qk", "av", "dq", "dv"))


@pytest.mark.gpu
@pytest.mark.parametrize("heads_first", [False, True])
@pytest.mark.parametrize("case", BIAS, ids=[f"{'x'.join(map(str, c[1]))}-k{c[4]}d{c[5]}" for c in BIAS])
def test_bias_gradient_partials(case, heads_first):
    """The workspace is NaN beforehand, so a partial that is not written shows.
    Sums are float64 throughout: only the result's rounding to float32 (2^-24)
    remains, and 2^-44 of the summed magnitudes for the order of the sum."""
    from natten_amd._core import hip

    B, sp, H, D, K, d = case
    print(f"[case] bias partials {case} heads_first={heads_first}", flush=True)
    r = len(sp)
    q, k = (randn((B, *sp, H, D), F32, i) for i in range(2))
    rpb = torch.zeros((H, *(2 * K - 1,) * r))
    gl = randn((B, *sp, H, K**r), F32, 3)
    ref = O.grads(lambda b: O.qk_rpb(q, k, b, K, d, 0.3), (rpb,), (gl,))[0]
    mag = O.grads(lambda b: O.qk_rpb(q, k, b, K, d, 0.3), (rpb,), (gl.abs(),))[0]
    put = (lambda t: t.movedim(-2, 1).contiguous().to(DEV)) if heads_first else (lambda t: t.to(DEV))
    qd, kd, gd = put(q), put(k), put(gl)
    lib = hip._lib.load()
    p = hip._rpb_params(qd, K, d, heads_first, 0.3)
    ws = torch.full((lib.na_rpb_bwd_workspace_bytes(p) // 8,), float("nan"), dtype=torch.float64,
                    device=DEV)
    dq, dk, drpb = torch.empty_like(qd), torch.empty_like(kd), torch.empty_like(rpb, device=DEV)
    P = hip._lib.ptr
    hip._lib.check(lib.na_rpb_qk_bwd(p, P(qd), P(kd), P(gd), P(dq), P(dk), P(drpb), P(ws),
                                     ws.numel() * 8, hip._lib.stream_of(qd)), "na_rpb_qk_bwd")
    err = (drpb.cpu().double() - ref).abs()
    assert bool((err <= 2.0**-24 * ref.abs() + 2.0**-44 * mag).all()), err.max()
