"""Weight and bias gradient kernels of the layers' projections (na_linear.hip)
against float64 sums, and the layer against torch's own linear backward."""

import pytest
import torch

from _helpers import DEV, randn

pytestmark = pytest.mark.gpu

BF16, F16 = torch.bfloat16, torch.float16


def _rel(a, b):
    return ((a.double() - b).norm() / b.norm()).item()


# rows around a stage of 64 and a split's 256, columns around a tile of 128
@pytest.mark.parametrize("dtype", [BF16, F16], ids=str)
@pytest.mark.parametrize("rows,n,k", [(1, 8, 8), (63, 128, 136), (65, 120, 128), (257, 8, 264),
                                      (1000, 392, 56), (5000, 96, 32), (4097, 256, 256)])
def test_weight_gradient(dtype, rows, n, k):
    from natten_amd._core import _lib

    lib, code = _lib.load(), _lib.dtype_code(dtype)
    g, x = randn((rows, n), dtype, 1).to(DEV), randn((rows, k), dtype, 2).to(DEV)
    dw = torch.full((n, k), float("nan"), dtype=dtype, device=DEV)
    db = torch.full((n,), float("nan"), dtype=dtype, device=DEV)
    nbytes = lib.na_linear_wgrad_workspace_bytes(code, rows, n, k)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
    eps = {BF16: 2.0 ** -8, F16: 2.0 ** -11}[dtype]  # one rounding of the result
    for bias in (db, None):
        _lib.check(lib.na_linear_wgrad(code, rows, n, k, g.data_ptr(), x.data_ptr(),
                                       dw.data_ptr(), _lib.ptr(bias), ws.data_ptr(), nbytes,
                                       _lib.stream_of(g)), "na_linear_wgrad")
        assert _rel(dw, g.double().t() @ x.double()) < eps
    assert _rel(db, g.double().sum(0)) < eps


def _layer(kv=None, dtype=BF16, bias=True):
    import natten_amd

    torch.manual_seed(0)
    return natten_amd.NeighborhoodAttention2D(64, 2, 5, num_kv_heads=kv, qkv_bias=bias).to(
        DEV, dtype)


@pytest.mark.parametrize("kv,bias", [(None, True), (1, True), (None, False)])
def test_layer_matches_torch_linear(kv, bias):
    import natten_amd.autograd.fused as AF

    m = _layer(kv, bias=bias)
    x = randn((2, 33, 31, 64), BF16, 3).to(DEV).requires_grad_(True)
    g = randn((2, 33, 31, 64), BF16, 4).to(DEV)
    leaves = [x, *m.parameters()]
    out = m(x)
    assert "CppNode" in out.grad_fn.name()
    a = [out, *torch.autograd.grad(out, leaves, g)]
    with AF.python_autograd():
        out = m(x)
        b = [out, *torch.autograd.grad(out, leaves, g)]
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])  # output and dx: torch's products
    for p, q in zip(a[2:], b[2:]):
        assert p.dtype == q.dtype and p.shape == q.shape
        assert _rel(p, q.double()) < 2.0 ** -8


def test_what_is_not_plain_keeps_the_module_call():
    m = _layer()
    x = randn((2, 33, 31, 64), BF16, 3).to(DEV)
    seen = []
    h = m.qkv.register_forward_hook(lambda *_: seen.append("hook"))
    m(x)
    h.remove()
    assert seen == ["hook"]

    def called(fn):
        real, calls = torch.nn.functional.linear, []
        torch.nn.functional.linear = lambda *a, **k: (calls.append(1), real(*a, **k))[1]
        try:
            fn()
        finally:
            torch.nn.functional.linear = real
        return len(calls)

    assert called(lambda: m(x)) == 0
    with torch.no_grad():
        assert called(lambda: m(x)) == 2
    with torch.autocast("cuda", dtype=F16):
        assert called(lambda: m(x)) == 2
    assert called(lambda: m(x[:1, :9, :9])) == 2          # few rows
    m.proj.weight.requires_grad_(False)
    assert called(lambda: m(x)) == 1                       # a frozen projection
    m.proj.weight.requires_grad_(True)
    # a backward that records a graph differentiates through the projections
    y = torch.nn.functional.silu(m.qkv(x)).sum()
    from natten_amd.nn import _linear

    z = torch.nn.functional.silu(_linear(m.qkv, x)).sum()
    second = []
    for v in (y, z):
        (gw,) = torch.autograd.grad(v, m.qkv.weight, create_graph=True)
        second.append(torch.autograd.grad(gw.float().square().sum(), m.qkv.weight)[0])
    assert _rel(second[1], second[0].double()) < 2.0 ** -6  # bf16 products in another order


@pytest.mark.parametrize("dtype,rank,sp,dim,heads,kw", [
    (torch.float32, 1, (70,), 48, 3, dict(kernel_size=7, stride=2)),
    (torch.float32, 2, (9, 11), 4, 1, dict(kernel_size=3)),           # one 16-byte unit a row
    (torch.float32, 2, (9, 11), 6, 2, dict(kernel_size=3)),           # not whole units: parts
    (BF16, 2, (17, 15), 64, 2, dict(kernel_size=5, dilation=2)),
    (F16, 3, (5, 8, 9), 32, 1, dict(kernel_size=3, is_causal=(True, False, False))),
    (BF16, 1, (33,), 128, 2, dict(kernel_size=33)),                   # dense
], ids=str)
def test_packed_projection_matches_parts(dtype, rank, sp, dim, heads, kw):
    import natten_amd
    import natten_amd.autograd.fused as AF

    torch.manual_seed(1)
    m = getattr(natten_amd, f"NeighborhoodAttention{rank}D")(dim, heads, **kw).to(DEV, dtype)
    for batch in (2, 0):
        x = randn((batch, *sp, dim), dtype, 5).to(DEV).requires_grad_(True)
        res = []
        for py in (False, True):
            with AF.python_autograd(py):
                out = m(x)
                g = randn(out.shape, dtype, 6).to(DEV)
                res.append([out, *torch.autograd.grad(out, [x, *m.parameters()], g)])
        for a, b in zip(*res):
            assert a.shape == b.shape and torch.equal(a, b)
