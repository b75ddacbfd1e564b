"""GPU tests of the backward on row tiles where the tiles of several sequences take turns in the list: few heads, so that up to eight sequences
form a group.  Against the float64 oracle on some heads, bit for bit against itself and against the same call without a prepared schedule
(the scheduler kernel lists each sequence's tiles together: the same sums in the same order)."""
import numpy as np
import pytest
import torch

from oracle import sb_oracle as orc
from stickbreaking_attention import _native, sb_attn, sb_attn_varlen
from test_gpu_parity import tol_check

pytestmark = pytest.mark.gpu

CASES = [      # heads, lengths (from 64 K rows x heads on the kernel runs)
    (12, [2048, 1025, 1024, 769, 512, 257, 1, 256, 255]),
    (8, [1500] * 6),
    (9, [3000, 0, 2000, 700, 700, 650, 300, 40, 33, 600]),
    (32, [700, 513, 512, 257, 300]),
]


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H,lengths", CASES, ids=[str(c[0]) for c in CASES])
@pytest.mark.parametrize("fixed", [False, True])
def test_against_oracle_and_the_plain_order(gpu_device, H, lengths, D, fixed):
    if fixed:
        lengths = [max(lengths[0], 1024)] * (70000 // (H * max(lengths[0], 1024)) + 1)
    T = sum(lengths)
    assert T * H >= 64 << 10
    g = torch.Generator().manual_seed(H + D)
    host = [torch.randn(H, T, D, generator=g).bfloat16() for _ in range(4)] + [torch.randn(H, T, generator=g).bfloat16()]
    dev = [t.to(gpu_device) for t in host]
    cu = torch.tensor(np.cumsum(lengths), dtype=torch.int32)

    def run():
        q, k, v = (t.detach().requires_grad_() for t in dev[:3])
        if fixed:
            def batched(t):
                return t.unflatten(1, (len(lengths), lengths[0])).transpose(0, 1)

            o, rem = sb_attn(batched(q), batched(k), batched(v))
            return torch.autograd.grad([o, rem], [q, k, v], [batched(dev[3]), batched(dev[4])])
        o, rem = sb_attn_varlen(q, k, v, cu if H == 9 else cu.to(gpu_device), max(lengths), zero_start=False)
        return torch.autograd.grad([o, rem], [q, k, v], dev[3:])

    saved = _native.POISON
    try:
        _native.POISON = True
        got, again = run(), run()
        _native.set_backward_workspace_limit(1 << 40)      # (nothing is prepared)
        plain = run()
    finally:
        _native.POISON = saved
        _native.set_backward_workspace_limit(None)
    heads = sorted({0, H - 1})
    ref = orc.varlen_stream(*(t[heads] for t in host[:3]), cu, do=host[3][heads], drem=host[4][heads], dtype=torch.float64)[2:]
    for name, a, b, c, r in zip(("dq", "dk", "dv"), got, again, plain, ref):
        assert torch.equal(a, b) and torch.equal(a, c), name
        tol_check(name, a[heads], r, torch.bfloat16, f"H={H} D={D} fixed={fixed}")


APART = [      # heads, lengths: sequences of one tile beside chains, listed by the forward (up to 64 sequences) and by the scheduler kernel
    (8, [4096] + [64] * 70),
    (12, [1025, 700, 300] + [255, 256, 1, 33] * 20),
    (32, [257] + [100] * 40),
    (9, [2000, 1500, 600] + [200] * 25),
    (32, [60] * 80),
]


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H,lengths", APART, ids=[f"{c[0]}x{len(c[1])}" for c in APART])
def test_sequences_of_one_tile_beside_chains(gpu_device, H, lengths, D):
    """A share of the workgroups begins with the sequences of a single tile: every tile is taken once whichever list is used up first."""
    T = sum(lengths)
    assert T * H >= 64 << 10
    g = torch.Generator().manual_seed(H + D)
    order = torch.randperm(len(lengths), generator=g).tolist()
    lengths = [lengths[i] for i in order]
    host = [torch.randn(H, T, D, generator=g).bfloat16() for _ in range(4)] + [torch.randn(H, T, generator=g).bfloat16()]
    dev = [t.to(gpu_device) for t in host]
    cu = torch.tensor(np.cumsum(lengths), dtype=torch.int32)

    def run():
        q, k, v = (t.detach().requires_grad_() for t in dev[:3])
        o, rem = sb_attn_varlen(q, k, v, cu if H == 9 else cu.to(gpu_device), max(lengths), zero_start=False)
        return torch.autograd.grad([o, rem], [q, k, v], dev[3:])

    saved = _native.POISON
    try:
        _native.POISON = True
        got, again = run(), run()
    finally:
        _native.POISON = saved
    heads = sorted({0, H - 1})
    ref = orc.varlen_stream(*(t[heads] for t in host[:3]), cu, do=host[3][heads], drem=host[4][heads], dtype=torch.float64)[2:]
    for name, a, b, r in zip(("dq", "dk", "dv"), got, again, ref):
        assert torch.equal(a, b), name
        tol_check(name, a[heads], r, torch.bfloat16, f"H={H} D={D}")
