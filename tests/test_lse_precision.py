"""16-bit fused forwards of row slabs and of samples of 2^24 elements or more:
their log-sum-exp holds a float32 row sum (MI355X)."""

import math

import pytest
import torch

from _helpers import DEV, randn

F16, BF16 = torch.float16, torch.bfloat16

# dtype, B, spatial, H, Hkv, D, kernel, dilation, causal
CASES = [
    (F16, 2, (96, 96), 8, 8, 64, (9, 9), (1, 1), (False, False)),      # row slabs
    (BF16, 1, (131, 75), 8, 4, 128, (5, 7), (1, 1), (True, False)),
    (BF16, 4, (112, 67), 4, 4, 32, (13, 11), (1, 1), (False, True)),
    (F16, 1, (523, 512), 2, 1, 32, (3, 5), (2, 1), (False, False)),    # 2^24 elements or more
    (BF16, 1, (371, 368), 2, 2, 64, (13, 3), (1, 1), (False, False)),
    (F16, 1, (132000,), 4, 2, 32, (7,), (1,), (True,)),
    (BF16, 1, (65536,), 4, 4, 64, (31,), (3,), (False,)),
    (F16, 1, (131072,), 1, 1, 128, (3,), (1,), (False,)),
]


def _lse(q, k, ks, dil, caus):
    """float64 log-sum-exp [B, tokens, H] of scaled window scores."""
    B, sp, H, D = q.shape[0], q.shape[1:-2], q.shape[-2], q.shape[-1]
    rep = H // k.shape[-2]
    tok = torch.zeros((1, 1), dtype=torch.int64, device=DEV)  # [queries, slots]
    good = torch.ones((1, 1), dtype=torch.bool, device=DEV)
    for n, K, d, c in zip(sp, ks, dil, caus):
        p = torch.arange(n, device=DEV)
        r, i = p % d, p // d
        size = (n - r + d - 1) // d
        first = i - K + 1 if c else torch.minimum((i - K // 2).clamp(min=0), size - K)
        j = first[:, None] + torch.arange(K, device=DEV)
        pos, ok = r[:, None] + d * j.clamp(min=0), j >= 0
        tok = (tok[:, None, :, None] * n + pos[None, :, None, :]).reshape(tok.shape[0] * n, -1)
        good = (good[:, None, :, None] & ok[None, :, None, :]).reshape(tok.shape)
    qf, kf = q.double().reshape(B, -1, H, D), k.double().reshape(B, -1, H // rep, D)
    s = torch.stack([(qf * kf[:, t].repeat_interleave(rep, 2)).sum(-1) for t in tok.T], -1)
    return torch.logsumexp((s * D ** -0.5).masked_fill(~good[None, :, None], -math.inf), -1)


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=[f"{'x'.join(map(str, c[2]))}-d{c[5]}" for c in CASES])
def test_row_sums_are_float32(case):
    from natten_amd._core import hip

    dtype, B, sp, H, Hkv, D, ks, dil, caus = case
    print(f"[case] lse {case}", flush=True)
    q = randn((B, *sp, H, D), dtype, 1).to(DEV)
    k, v = (randn((B, *sp, Hkv, D), dtype, i).to(DEV) for i in (2, 3))
    with hip.any_size_kernels():
        _, lse = hip.fused_forward(q, k, v, ks, (1,) * len(sp), dil, caus, None)
    err = (lse.double().reshape(B, -1, H) - _lse(q, k, ks, dil, caus)).abs().max()
    # a probability: 2^-21 (its rounded exponent below 16) + 2^-22 (exp2); a
    # lane's sum of at most 64: 2^-18; the scores' sums over head_dim, times
    # the score's size below 8: 2^-18; the value itself, below 8: 2^-21.  One
    # probability rounded to 16 bits would add up to 2^-12.
    assert float(err) < 1e-5, float(err)
