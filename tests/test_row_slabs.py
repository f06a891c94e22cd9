"""Rank-2 lean kernels whose box is staged a few rows at a time: the plan (CPU),
and forward + LSE + backward against the oracle at the edges of slabs, tiles and
images (MI355X)."""

import pytest
import torch

from _helpers import DEV, assert_close, randn
from oracle import na as O

F16, BF16 = torch.float16, torch.bfloat16


def _plan(B, sp, H, Hkv, D, ks, dil, caus, dtype, backward):
    from natten_amd._core import hip

    q = torch.empty((B, *sp, H, D), dtype=dtype, device="meta")
    k = torch.empty((B, *sp, Hkv, D), dtype=dtype, device="meta")
    return hip.kernel_plan(q, k, ks, (1, 1), dil, caus, backward=backward)


def test_large_images_and_sequences_run_lean():
    """The 24-bit stride limit is on the axes a problem has, not on the unit
    axes before them."""
    for sp, H, D, ks in (((384, 384), 8, 64, (7, 7)), ((256, 256), 16, 64, (7, 7)),
                         ((65536,), 16, 64, (63,))):
        from natten_amd._core import hip

        q = torch.empty((1, *sp, H, D), dtype=F16, device="meta")
        one, no = (1,) * len(sp), (False,) * len(sp)
        for backward in (False, True):
            assert hip.kernel_path(q, q, ks, one, one, no, backward=backward) == "lean"


# (dtype, B, spatial, H, Hkv, D, kernel, dilation, causal)
CASES = [
    (F16, 1, (20, 19), 2, 1, 64, (13, 13), (1, 1), (False, False)),   # two-chunk inverse rows
    (F16, 1, (33, 17), 1, 1, 64, (13, 9), (1, 1), (True, False)),
    (BF16, 1, (49, 56), 2, 2, 64, (11, 11), (2, 3), (False, False)),  # phases of unequal length
    (BF16, 2, (14, 23), 2, 1, 128, (7, 7), (1, 1), (False, False)),
    (F16, 1, (19, 16), 4, 1, 128, (5, 7), (1, 1), (False, True)),     # four heads per box
    (F16, 1, (9, 13), 1, 1, 128, (9, 13), (1, 1), (False, True)),     # window = image
    (BF16, 1, (18, 35), 1, 1, 128, (13, 13), (1, 1), (False, False)),
]


@pytest.mark.parametrize("case", CASES, ids=[f"{c[2]}-d{c[5]}-k{c[6]}" for c in CASES])
def test_planned_in_row_slabs(case):
    from natten_amd._core import hip

    with hip.any_size_kernels():  # small launches: see the rules below
        p = _plan(*case[1:], case[0], True)
    assert p["path"] == "lean" and p["slabs"] > 1, p


# What a launch's size and shape decide: (B, spatial, H, Hkv, D, kernel, backward)
# and the plan: path, boxes in slabs, waves.
LAUNCHES = [
    # too few workgroups, or many query heads to one: not in slabs
    ((1, (27, 36), 16, 1, 64, (15, 15), True), ("mfma", False)),
    ((4, (56, 56), 16, 2, 32, (13, 13), True), ("mfma", False)),
    ((1, (43, 27), 4, 1, 128, (5, 5), True), ("lean", False)),
    ((1, (74, 52), 2, 2, 64, (7, 7), False), ("lean", False)),
    ((2, (23, 26), 1, 1, 64, (11, 7), False), ("lean", False)),
    ((4, (56, 56), 4, 4, 32, (13, 13), False), ("lean", False)),
    # a row of 17 padded to 32; a large image's two-wave boxes
    ((1, (290, 420), 1, 1, 64, (11, 11), True), ("mfma", False)),
    ((2, (306, 351), 4, 4, 64, (5, 9), True), ("mfma", False)),
    # enough of them
    ((2, (96, 96), 8, 8, 64, (9, 9), True), ("lean", True)),
    ((1, (256, 256), 16, 16, 128, (7, 7), True), ("lean", True)),
    ((2, (112, 112), 4, 4, 64, (5, 5), False), ("lean", True)),
    ((8, (91, 79), 16, 16, 32, (13, 13), False), ("lean", True)),  # 32 per CU and more
    ((2, (72, 100), 8, 8, 128, (5, 5), False), ("lean", True)),
    # no whole box: the forward in slabs at any size
    ((1, (21, 20), 1, 1, 128, (13, 13), False), ("lean", True)),
]


@pytest.mark.parametrize("problem,want", LAUNCHES, ids=[f"{c[0]}" for c in LAUNCHES])
def test_slabs_where_the_launch_gains(problem, want):
    B, sp, H, Hkv, D, ks, backward = problem
    p = _plan(B, sp, H, Hkv, D, ks, (1, 1), (False, False), F16, backward)
    assert (p["path"], p["slabs"] > 1) == want, p


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=[f"{c[2]}-d{c[5]}-k{c[6]}" for c in CASES])
def test_row_slabs_against_oracle(case):
    from natten_amd._core import hip

    with hip.any_size_kernels():
        _row_slabs_against_oracle(case)


def _row_slabs_against_oracle(case):
    import natten_amd

    dtype, B, sp, H, Hkv, D, ks, dil, caus = case
    print(f"[case] row slabs {case}", flush=True)
    q, k, v = (randn((B, *sp, h, D), dtype, i) for i, h in enumerate((H, Hkv, Hkv)))
    ts = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]
    out, lse = natten_amd.na2d(*ts, ks, 1, dil, caus, return_lse=True)

    def f(a, b, c):
        return O.na_functional(a, b, c, ks, 1, dil, caus, return_lse=True)

    ro, rl = f(q, k, v)
    assert_close(out, ro, dtype, "out")
    assert_close(lse, rl, dtype, "lse")
    go, gl = randn(out.shape, dtype, 7), randn(lse.shape, dtype, 8)
    torch.autograd.backward((out, lse), (go.to(DEV), gl.to(DEV)))
    for t, r, n in zip(ts, O.grads(f, (q, k, v), (go, gl)), ("dq", "dk", "dv")):
        assert_close(t.grad, r, dtype, n)


# Rank-3 boxes beyond LDS: eight waves on several layers.  (dtype, B, spatial, H,
# Hkv, D, kernel, dilation, causal), large enough for two workgroups per CU.
DEPTH = [
    (BF16, 2, (9, 34, 33), 8, 4, 32, (3, 7, 7), (1, 1, 1), (False, False, False)),
    (F16, 1, (11, 40, 40), 8, 8, 64, (3, 5, 5), (1, 1, 1), (True, False, False)),
    (BF16, 1, (10, 33, 41), 16, 4, 64, (3, 7, 7), (1, 1, 2), (False, True, False)),
]


@pytest.mark.parametrize("case", DEPTH, ids=[f"{c[2]}-d{c[5]}" for c in DEPTH])
def test_planned_on_several_layers(case):
    from natten_amd._core import hip

    dtype, B, sp, H, Hkv, D, ks, dil, caus = case
    q = torch.empty((B, *sp, H, D), dtype=dtype, device="meta")
    k = torch.empty((B, *sp, Hkv, D), dtype=dtype, device="meta")
    p = hip.kernel_plan(q, k, ks, (1, 1, 1), dil, caus)
    assert p["path"] == "lean" and p["waves"] == 8 and p["slabs"] == p["box"][0], p


# (B, spatial, H, Hkv, D, kernel, dilation, causal, backward) and waves per workgroup.
LAYERS = [
    # ragged tiles that add a third of waves, a second round of a few workgroups
    ((1, (9, 30, 38), 2, 2, 128, (3, 3, 3), 1, (True, False, False), False), 4),
    ((1, (9, 30, 38), 2, 2, 128, (3, 3, 3), 1, (True, False, False), True), 2),
    ((8, (20, 32, 19), 1, 1, 64, (7, 3, 3), 2, (True, False, False), False), 4),
    ((1, (10, 38, 28), 4, 4, 128, (7, 7, 7), (1, 2, 2), (False,) * 3, False), 4),
    # three four-wave workgroups to a CU
    ((2, (3, 21, 44), 16, 16, 32, (3, 7, 7), 1, (False,) * 3, True), 4),
    ((1, (16, 32, 32), 8, 8, 64, (3, 7, 7), 1, (True, False, False), False), 8),
    ((1, (16, 32, 32), 8, 8, 64, (3, 7, 7), 1, (True, False, False), True), 8),
]


@pytest.mark.parametrize("problem,waves", LAYERS, ids=[f"{c[0][1]}-{c[0][8]}" for c in LAYERS])
def test_layers_where_the_launch_gains(problem, waves):
    from natten_amd._core import hip

    B, sp, H, Hkv, D, ks, dil, caus, backward = problem
    q = torch.empty((B, *sp, H, D), dtype=BF16, device="meta")
    k = torch.empty((B, *sp, Hkv, D), dtype=BF16, device="meta")
    dil = (dil,) * 3 if isinstance(dil, int) else dil
    p = hip.kernel_plan(q, k, ks, (1, 1, 1), dil, caus, backward=backward)
    assert p["path"] == "lean" and p["waves"] == waves, p


@pytest.mark.gpu
@pytest.mark.parametrize("case", DEPTH, ids=[f"{c[2]}-d{c[5]}" for c in DEPTH])
def test_several_layers_against_the_32_query_kernels(case):
    import natten_amd
    from natten_amd._core import hip

    dtype, B, sp, H, Hkv, D, ks, dil, caus = case
    print(f"[case] several layers {case}", flush=True)
    ts = [randn((B, *sp, h, D), dtype, i).to(DEV).requires_grad_(True)
          for i, h in enumerate((H, Hkv, Hkv))]
    res = []
    for other in (False, True):
        with hip.no_lean_kernels(other):
            out, lse = natten_amd.na3d(*ts, ks, 1, dil, caus, return_lse=True)
            go = randn(out.shape, dtype, 7).to(DEV)
            gl = randn(lse.shape, dtype, 8).to(DEV)
            res.append([out, lse, *torch.autograd.grad((out, lse), ts, (go, gl))])
    for a, b, n in zip(*res, ("out", "lse", "dq", "dk", "dv")):
        assert_close(a, b.double(), dtype, n)
