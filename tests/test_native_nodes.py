"""The split and DiNAT operators' C++ autograd nodes against the Python
Functions over the same kernels, bit for bit: mixed and 16-bit types,
non-contiguous inputs, partial gradients, saved-tensor hooks, side streams and
graph capture; and what they refuse."""

import pytest
import torch

from _helpers import DEV, randn

F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16


def _split(ts, arg):
    from natten_amd import functional as F

    q, k, v = ts
    r = q.dim() - 3
    logits = getattr(F, f"na{r}d_qk")(q, k, **arg)
    attn = torch.softmax(logits, -1)
    return logits, getattr(F, f"na{r}d_av")(attn, v, **arg)


def _rpb(ts, arg):
    from natten_amd.autograd.allin1 import av_rpb_with_grad, qk_rpb_with_grad

    q, k, v, rpb = (*ts, None)[:4]
    K, d = arg["kernel_size"], arg["dilation"]
    logits = qk_rpb_with_grad(q, k, rpb, K, d, arg.get("scale"), arg.get("heads_first", False))
    out = av_rpb_with_grad(torch.softmax(logits, -1), v, K, d, arg.get("heads_first", False),
                           arg.get("out_dtype", F32))
    return logits, out


def _t(shape, dt, seed):
    return randn(shape, dt, seed).to(DEV)


CASES = {
    "split 1d f32": (_split, [((2, 40, 4, 32), F32)] * 3, dict(kernel_size=7, dilation=2)),
    "split 2d bf16": (_split, [((1, 12, 14, 4, 32), BF16)] * 3, dict(kernel_size=(7, 5))),
    "split 2d gqa": (_split, [((1, 12, 14, 4, 32), F16)] + [((1, 12, 14, 2, 32), F16)] * 2,
                     dict(kernel_size=3, stride=2)),
    "split 3d causal": (_split, [((1, 4, 6, 7, 2, 16), F32)] * 3,
                        dict(kernel_size=3, is_causal=(True, False, False))),
    "split mixed types": (_split, [((1, 9, 9, 2, 32), F32), ((1, 9, 9, 2, 32), BF16),
                                   ((1, 9, 9, 2, 32), F16)], dict(kernel_size=3)),
    "rpb 1d": (_rpb, [((2, 50, 3, 12), F32)] * 3 + [((3, 13), F32)],
               dict(kernel_size=7, dilation=2, scale=0.288)),
    "rpb 2d": (_rpb, [((1, 15, 14, 2, 32), F32)] * 3 + [((2, 9, 9), F32)],
               dict(kernel_size=5, dilation=2)),
    "rpb 2d no bias": (_rpb, [((1, 9, 10, 2, 16), F32)] * 3, dict(kernel_size=3, dilation=1)),
    "rpb heads first": (_rpb, [((1, 2, 14, 15, 16), F32)] * 3 + [((2, 5, 9), F32)],
                        dict(kernel_size=(3, 5), dilation=(2, 1), heads_first=True)),
    "rpb bf16": (_rpb, [((1, 30, 2, 12), BF16)] * 3 + [((2, 9), BF16)],
                 dict(kernel_size=5, dilation=1, out_dtype=BF16, scale=0.3)),
}


def _run(case, need=None, transpose=False):
    fn, shapes, arg = CASES[case]
    ts = [_t(s, dt, i) for i, (s, dt) in enumerate(shapes)]
    if transpose:
        ts = [t.transpose(0, -1).contiguous().transpose(0, -1) for t in ts]
    need = need or [True] * len(ts)
    ts = [t.requires_grad_(n) for t, n in zip(ts, need)]
    logits, out = fn(ts, arg)
    g = _t(out.shape, out.dtype, 9)
    leaves = [t for t in ts if t.requires_grad]
    return [logits, out, *torch.autograd.grad(out, leaves, g)]


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(CASES))
def test_nodes_match_python_functions(case):
    import natten_amd.autograd.fused as AF

    n = len(CASES[case][1])
    for need, tr in ((None, False), (None, True), ([i == 2 for i in range(n)], False),
                     ([i == 0 for i in range(n)], False)):
        a = _run(case, need, tr)
        with AF.python_autograd():
            b = _run(case, need, tr)
        assert "CppNode" in a[1].grad_fn.name() and "CppNode" not in b[1].grad_fn.name()
        for x, y in zip(a, b):
            assert x.dtype == y.dtype and x.shape == y.shape and torch.equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["split 2d bf16", "rpb 2d"])
def test_nodes_hooks_streams_and_capture(case):
    want = _run(case)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t.cpu(),
                                                  lambda t: t.to(DEV)):
        got = _run(case)
    assert len(packed) >= 4
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        other = _run(case)
    torch.cuda.current_stream().wait_stream(side)
    for x, y, z in zip(want, got, other):
        assert torch.equal(x, y) and torch.equal(x, z)

    fn, shapes, arg = CASES[case]
    ts = [_t(s, dt, i).requires_grad_(True) for i, (s, dt) in enumerate(shapes)]
    g = _t(want[1].shape, want[1].dtype, 9)

    def step():
        out = fn(ts, arg)[1]
        return [out, *torch.autograd.grad(out, ts, g)]

    with torch.cuda.stream(side):
        step()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            res = step()
    for _ in range(3):
        for t in res:
            t.detach().zero_()
        graph.replay()
        torch.cuda.synchronize()
        for x, y in zip(res, want[1:]):
            assert torch.equal(x, y)
        step()


def _ops():
    from natten_amd._core import _lib

    _lib.load()
    return torch.ops.natten_amd


# Direct calls of the operators on CPU tensors: (operator, arguments, message).  The
# shapes are checked on the host before the device is.
_z = torch.zeros
_HIP = "HIP"
DIRECT = [
    ("na_split_qk", (_z(1, 9, 9, 4, 32), _z(1, 9, 9, 2, 32), [3, 3], [1, 1], [1, 1], [0, 0], 1.0, 0), _HIP),
    ("na_split_qk", (_z(1, 9, 9, 4, 32), _z(1, 9, 8, 2, 32), [3, 3], [1, 1], [1, 1], [0, 0], 1.0, 0), "q .B"),
    ("na_split_qk", (_z(2, 9, 9, 4, 32), _z(1, 9, 9, 4, 32), [3, 3], [1, 1], [1, 1], [0, 0], 1.0, 0), "q .B"),
    ("na_split_qk", (_z(1, 9, 9, 4, 32), _z(1, 9, 9, 3, 32), [3, 3], [1, 1], [1, 1], [0, 0], 1.0, 0), "q .B"),
    ("na_split_qk", (_z(1, 9, 9, 4, 32), _z(1, 9, 9, 4, 16), [3, 3], [1, 1], [1, 1], [0, 0], 1.0, 0), "q .B"),
    ("na_split_qk", (_z(1, 9, 9, 4, 32), _z(1, 9, 4, 32), [3, 3], [1, 1], [1, 1], [0, 0], 1.0, 0), "q .B"),
    ("na_split_qk", (_z(1, 9, 9, 4, 32), _z(1, 9, 9, 4, 32), [3], [1], [1], [0], 1.0, 0), "per spatial axis"),
    ("na_split_qk", (_z(1, 9, 9, 4, 32), _z(1, 9, 9, 4, 32), [3, 3], [1, 0], [1, 1], [0, 0], 1.0, 0), "positive"),
    ("na_split_av", (_z(1, 5, 9, 4, 9), _z(1, 9, 9, 2, 32), [3, 3], [2, 1], [1, 1], [0, 0]), _HIP),
    ("na_split_av", (_z(1, 4, 9, 4, 9), _z(1, 9, 9, 2, 32), [3, 3], [2, 1], [1, 1], [0, 0]), "attn is"),
    ("na_split_av", (_z(1, 9, 9, 4, 8), _z(1, 9, 9, 2, 32), [3, 3], [1, 1], [1, 1], [0, 0]), "attn is"),
    ("na_split_av", (_z(2, 9, 9, 4, 9), _z(1, 9, 9, 2, 32), [3, 3], [1, 1], [1, 1], [0, 0]), "attn is"),
    ("na_split_av", (_z(1, 9, 9, 3, 9), _z(1, 9, 9, 2, 32), [3, 3], [1, 1], [1, 1], [0, 0]), "attn is"),
    ("na_split_av", (_z(1, 9, 4, 9), _z(1, 9, 9, 2, 32), [3, 3], [1, 1], [1, 1], [0, 0]), "attn is"),
    ("na_rpb_qk", (_z(1, 9, 8, 2, 32), _z(1, 9, 8, 2, 32), _z(2, 5, 5), [3, 3], [1, 1], 1.0, True, False), _HIP),
    ("na_rpb_qk", (_z(1, 9, 8, 2, 32), _z(1, 9, 8, 2, 32), _z(2, 5, 3), [3, 3], [1, 1], 1.0, True, False), "rpb must"),
    ("na_rpb_qk", (_z(1, 9, 8, 2, 32), _z(1, 9, 8, 2, 32), _z(2, 5, 5), [3, 3], [1, 1], 1.0, True, True), "rpb must"),
    ("na_rpb_qk", (_z(1, 9, 8, 2, 32), _z(1, 8, 8, 2, 32), None, [3, 3], [1, 1], 1.0, True, False), "identical"),
    ("na_rpb_qk", (_z(1, 9, 2, 32), _z(1, 9, 2, 32), None, [3, 3], [1, 1], 1.0, True, False), "rank-1 or rank-2"),
    ("na_rpb_av", (_z(1, 9, 8, 2, 9), _z(1, 9, 8, 2, 32), [3, 3], [1, 1], False, True), _HIP),
    ("na_rpb_av", (_z(1, 9, 8, 2, 8), _z(1, 9, 8, 2, 32), [3, 3], [1, 1], False, True), "attn must"),
    ("na_rpb_av", (_z(1, 8, 9, 2, 9), _z(1, 9, 8, 2, 32), [3, 3], [1, 1], False, True), "attn must"),
    ("na_rpb_av", (_z(1, 9, 8, 2, 9), _z(1, 9, 8, 2, 32), [3, -3], [1, 1], False, True), "positive"),
    ("na_fused_qkv", (_z(1, 9, 3, 2, 32), [3], [1], [1], [0], 1.0, 0), _HIP),
    ("na_fused_qkv", (_z(1, 9, 2, 2, 32), [3], [1], [1], [0], 1.0, 0), "qkv is"),
    ("na_fused_qkv", (_z(1, 9, 3, 2, 32), [3, 3], [1], [1], [0], 1.0, 0), "per spatial axis"),
    ("na_fused_qkv", (_z(1, 9, 3, 2, 32), [3], [0], [1], [0], 1.0, 0), "positive"),
    ("na_linear", (_z(5, 32), _z(16, 32), _z(16)), _HIP),
    ("na_linear", (_z(5, 32), _z(16, 24), None), "na_linear: x"),
    ("na_linear", (_z(5, 32), _z(16, 32), _z(1)), "na_linear: x"),
]


@pytest.mark.parametrize("name,args,message", DIRECT, ids=[f"{i}-{c[0]}" for i, c in enumerate(DIRECT)])
def test_direct_calls_check_shapes(name, args, message):
    """A kernel indexes by the sizes of one tensor of a call: a mismatched call
    raises before any launch."""
    with pytest.raises(RuntimeError, match=message):
        getattr(_ops(), name)(*args, 0)


@pytest.mark.gpu
def test_nodes_refuse_what_the_functions_refuse():
    from natten_amd import functional as F
    from natten_amd.extras import allin1

    q = _t((1, 9, 9, 2, 32), F32, 0)
    attn = torch.softmax(F.na2d_qk(q, q, 3), -1)
    with pytest.raises(ValueError):
        F.na2d_av(attn, q, 5)                        # 9 slots, not 25
    with pytest.raises(ValueError):
        F.na2d_qk(q, q, 11)                          # larger than the image
    with pytest.raises(TypeError):
        F.na2d_qk(q.double(), q.double(), 3)
    with pytest.raises(RuntimeError):
        F.na2d_qk(q, q.cpu(), 3)
    with pytest.raises(RuntimeError):
        F.na2d_qk(q.cpu(), q.cpu(), 3)
    with pytest.raises(ValueError):
        allin1.na2d_qk_rpb(q, q, _t((2, 3, 5), F32, 1), 3)   # bias of another window
    with pytest.raises(ValueError):
        allin1.na2d_qk_rpb(q, q[:, :8], None, 3)
    with pytest.raises(ValueError):
        allin1.na2d_av_fused(attn, q, 5)
    empty = q[:0].requires_grad_(True)
    out = F.na2d_av(torch.softmax(F.na2d_qk(empty, empty, 3), -1), empty, 3)
    assert out.shape == (0, 9, 9, 2, 32)
    assert torch.autograd.grad(out.sum(), empty)[0].shape == empty.shape


@pytest.mark.gpu
def test_compiled_split_ops_run_as_eager():
    """The operators have no fake kernels: under compilation the split ops are
    Python Functions left to eager execution."""
    import natten_amd

    torch.manual_seed(0)
    layer = natten_amd.NeighborhoodAttention2D(64, 2, 3, attn_drop=0.1).to(DEV).eval()
    x = _t((1, 12, 14, 64), F32, 1).requires_grad_()
    ts = [_t((1, 12, 14, 2, 32), F32, i).requires_grad_() for i in range(3)]
    for fn, leaves in ((lambda *a: _split(a, dict(kernel_size=3))[1], ts), (layer, [x])):
        torch._dynamo.reset()
        res = []
        for f in (fn, torch.compile(fn, backend="eager")):
            out = f(*leaves)
            res.append([out, *torch.autograd.grad(out.square().sum(), leaves)])
        for a, b in zip(*res):
            assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["split 2d bf16", "rpb 1d"])
def test_transforms_stay_refused(case):
    fn, shapes, arg = CASES[case]
    ts = [_t(s, dt, i) for i, (s, dt) in enumerate(shapes)]
    with pytest.raises(RuntimeError, match="functorch"):
        torch.vmap(lambda *a: fn(a, arg)[1])(*[t[None].repeat(2, *[1] * t.dim()) for t in ts])
    with pytest.raises(RuntimeError, match="functorch"):
        torch.func.grad(lambda *a: fn(a, arg)[1].float().sum())(*ts)
    with torch.autograd.forward_ad.dual_level(), pytest.raises(NotImplementedError):
        fn([torch.autograd.forward_ad.make_dual(t, torch.ones_like(t)) for t in ts], arg)
