"""GPU tests of the backward on row tiles where the tiles of several sequences take turns in the list (few heads, so that up to eight sequences
form a group) and where those of sequences of one tile have a list of their own.  That a call runs there is asserted.  Against the float64 oracle on some heads, bit for bit against itself and against the same call without a prepared schedule
(the scheduler kernel lists each sequence's tiles together: the same sums in the same order)."""
import numpy as np
import pytest
import torch

from oracle import sb_oracle as orc
from stickbreaking_attention import _native, sb_attn, sb_attn_varlen
from test_gpu_backward_route import runs_on_row_tiles
from test_gpu_parity import tol_check

pytestmark = pytest.mark.gpu

CASES = [      # heads, lengths: groups of 2, 3, 4, 8 and 1 sequences, with an empty one, and with sequences of one tile beside longer ones
    (12, [1024, 1025, 769, 800, 900, 1000, 600, 513, 255]),
    (16, [1300, 900, 700, 257, 256, 1, 0, 1100]),
    (9, [1100, 1000, 900, 800, 700, 600, 513, 512, 300, 257, 1000, 0]),
    (8, [1500] * 6),
    (8, [2500, 0, 1800, 700, 513, 512, 300, 256, 40, 1500, 300]),
    (4, [2500, 2300, 2000, 1800, 1700, 1500, 1400, 1200, 900, 700, 300, 200]),
    (32, [700, 513, 512, 257, 300, 1000]),
]
OTHERS = [      # (some of these run on row tiles at equal lengths or at head_dim 128 only)
    (12, [2048, 1025, 1024, 769, 512, 257, 1, 256, 255]),
    (9, [3000, 0, 2000, 700, 700, 650, 300, 40, 33, 600]),
    (32, [700, 513, 512, 257, 300]),
]


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H,lengths", CASES + OTHERS, ids=[f"{c[0]}x{len(c[1])}" for c in CASES + OTHERS])
@pytest.mark.parametrize("fixed", [False, True])
def test_against_oracle_and_the_plain_order(gpu_device, H, lengths, D, fixed):
    listed = (H, lengths) in CASES
    if fixed:
        lengths = [max(lengths[0], 1024)] * max(8 if H & 7 else 1, 70000 // (H * max(lengths[0], 1024)) + 1)
    T = sum(lengths)
    assert T * H >= 64 << 10
    assert not listed or runs_on_row_tiles(H, D, lengths, fixed=fixed, lengths_known=H == 9)
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


APART = [      # heads, lengths: sequences of one tile beside one chain, listed by the forward (up to 64 sequences) and by the scheduler kernel
    (8, [4096] + [64] * 100),
    (8, [4000] + [250] * 40),
    (7, [4000] + [250] * 40),
    (16, [3000] + [200] * 20),
    (15, [3000, 260] + [150] * 45),
    (264, [250]),
    (300, [200, 20]),
]
TOGETHER = [      # ... and where one list holds all
    (12, [1025, 700, 300] + [255, 256, 1, 33] * 20),
    (32, [257] + [100] * 40),
    (32, [60] * 40 + [65] * 40),
    (8, [1024] + [60] * 200),
    (8, [4096] + [64] * 70),
]
KERNELS = [      # ... and for which the dQ and dK/dV kernels run
    (9, [2000, 1500, 600] + [200] * 25),
    (32, [60] * 80),
]


def work(n):
    return sum(-(-n // 32) - 8 * i + 1 for i in range(-(-n // 256)))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H,lengths,two", [(*c, c in APART) for c in APART + TOGETHER + KERNELS],
                         ids=[f"{c[0]}x{len(c[1])}" for c in APART + TOGETHER + KERNELS])
def test_sequences_of_one_tile_beside_chains(gpu_device, H, lengths, two, D):
    """A share of the workgroups begins with the sequences of a single tile: every tile is taken once whichever list is used up first.  (At
    head_dim 64 the kernel runs from a mean of 512 tokens on, where those are never a fifth of the work.)"""
    T = sum(lengths)
    assert T * H >= 64 << 10
    assert runs_on_row_tiles(H, D, lengths) == (D == 128 and (H, lengths) not in KERNELS)
    single, chained, longest = sum(work(n) for n in lengths if n <= 256), sum(work(n) for n in lengths if n > 256), max(map(work, lengths))
    total = single + chained
    assert two == (5 * single >= total and 3 * longest >= 2 * total and 16 * (chained - longest) <= total)
    g = torch.Generator().manual_seed(H + D)
    order = torch.randperm(len(lengths), generator=g).tolist()
    lengths = [lengths[i] for i in order]
    host = [torch.randn(H, T, D, generator=g).bfloat16() for _ in range(4)] + [torch.randn(H, T, generator=g).bfloat16()]
    dev = [t.to(gpu_device) for t in host]
    cu = torch.tensor(np.cumsum(lengths), dtype=torch.int32)

    def run(cu):
        q, k, v = (t.detach().requires_grad_() for t in dev[:3])
        o, rem = sb_attn_varlen(q, k, v, cu, max(lengths), zero_start=False)
        return torch.autograd.grad([o, rem], [q, k, v], dev[3:])

    saved = _native.POISON
    try:
        _native.POISON = True
        got, again, known = run(cu.to(gpu_device)), run(cu.to(gpu_device)), run(cu)
        _native.set_backward_workspace_limit(1 << 40)      # (listed by the scheduler kernel)
        plain = run(cu.to(gpu_device))
    finally:
        _native.POISON = saved
        _native.set_backward_workspace_limit(None)
    heads = sorted({0, H - 1})
    ref = orc.varlen_stream(*(t[heads] for t in host[:3]), cu, do=host[3][heads], drem=host[4][heads], dtype=torch.float64)[2:]
    for name, a, b, c, d, r in zip(("dq", "dk", "dv"), got, again, known, plain, ref):
        assert torch.equal(a, b) and torch.equal(a, c) and torch.equal(a, d), name
        tol_check(name, a[heads], r, torch.bfloat16, f"H={H} D={D}")
