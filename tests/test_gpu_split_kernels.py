"""The kernels of problems too small to fill the chip (keys split over the waves): lengths around their 32-row blocks and
128-key steps, rows no sequence covers, both directions, against the float64 oracle; and both kinds of kernel on the two sides
of the size from which on the wide ones run; and which of them runs when the lengths are known but max_seqlens is not given."""
import numpy as np
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from oracle import sb_oracle as orc
from stickbreaking_attention import sb_attn_varlen
from test_gpu_parity import NAMES, tol_check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("attend_current,add_remainder,save_carry", [(False, False, True), (True, True, False)])
@pytest.mark.parametrize("H,D", [(2, 24), (3, 64), (2, 100), (3, 128), (40, 64), (25, 128)])
def test_lengths_around_the_steps(gpu_device, H, D, attend_current, add_remainder, save_carry):
    lengths, pad = [1, 31, 32, 33, 95, 127, 128, 129, 160, 257, 300], 50
    dtype = torch.bfloat16
    T = sum(lengths)
    g = torch.Generator().manual_seed(H * D)
    host = [torch.randn(H, T + pad, D, generator=g).to(dtype) for _ in range(4)] + [torch.randn(H, T + pad, generator=g).to(dtype)]
    q, k, v, do, drem = (t.to(gpu_device) for t in host)
    for t in (q, k, v):
        t.requires_grad_()
    cu = torch.tensor(np.cumsum(lengths), dtype=torch.int32)
    o, rem = sb_attn_varlen(q, k, v, cu, max(lengths), zero_start=False, attend_current=attend_current, add_remainder=add_remainder,
                            save_carry=save_carry)
    got = (o, rem, *torch.autograd.grad([o, rem], [q, k, v], [do, drem]))
    heads = sorted({0, H - 1})
    d = [t[heads, :T].double() for t in host]
    if add_remainder:
        d[4] = orc.remainder_drem(d[3], d[4], d[2])
    ref = orc.varlen_stream(d[0], d[1], d[2], cu, attend_current=attend_current, do=d[3], drem=d[4], dtype=torch.float64)
    if add_remainder:
        ref = orc.with_remainder(ref, d[2], d[3])
    for n, a, b in zip(NAMES, got, ref):
        tol_check(n, a[heads, :T], b, dtype, f"H={H} D={D}")
        assert (a[:, T:] == 0).all(), f"{n}: rows no sequence covers must be zero"


@pytest.mark.parametrize("H,D", [(2, 50), (2, 64), (1, 128)])
@pytest.mark.parametrize("values", ["normal", "slow"])
def test_waves_with_several_sub_tiles(gpu_device, H, D, values):
    """Each wave of the forward sweeps a contiguous part of a row's keys, whose products are put on top of each other at the end: rows
    whose sub-tiles do not divide by the waves, sticks that end within a part and sticks that last over all of them."""
    lengths = [385, 513, 1000, 1441]
    T = sum(lengths)
    g = torch.Generator().manual_seed(H * D)
    q, k, v, do = (torch.randn(H, T, D, generator=g) for _ in range(4))
    if values == "slow":
        q, k = 0.25 * (q + 1), 0.25 * (k - 1)
    host = [t.bfloat16() for t in (q, k, v, do, torch.randn(H, T, generator=g))]
    q, k, v, do, drem = (t.to(gpu_device) for t in host)
    for t in (q, k, v):
        t.requires_grad_()
    cu = torch.tensor(np.cumsum(lengths), dtype=torch.int32)
    o, rem = sb_attn_varlen(q, k, v, cu, max(lengths), zero_start=False)
    got = (o, rem, *torch.autograd.grad([o, rem], [q, k, v], [do, drem]))
    ref = orc.varlen_stream(*(t.double() for t in host[:3]), cu, do=host[3].double(), drem=host[4].double(), dtype=torch.float64)
    for n, a, b in zip(NAMES, got, ref):
        tol_check(n, a, b, torch.bfloat16, f"H={H} D={D} {values}")


class Passing(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("where", ["host", "device with a leading zero", "host, Python operators"])
def test_known_lengths_choose_the_kernels_without_max_seqlens(gpu_device, where):
    """24 heads of 8 x 300 tokens: too many rows to split the keys of sequences this short, few enough if they were one.  The bits
    tell the kernels apart."""
    H, D, lengths = 24, 64, [300] * 8
    q, k, v, do = (torch.randn(H, sum(lengths), D, device=gpu_device).bfloat16() for _ in range(4))
    for t in (q, k, v):
        t.requires_grad_()
    zero = "zero" in where
    cu = torch.tensor(np.cumsum([0] * zero + lengths), dtype=torch.int32, device=gpu_device if zero else "cpu")

    def run(max_seqlens):
        o, rem = sb_attn_varlen(q, k, v, cu, max_seqlens, zero_start=zero)
        return o, rem, *torch.autograd.grad(o, [q, k, v], do)

    want = run(300)
    for hint in (None, 2000):
        if "operators" in where:
            with Passing():
                got = run(hint)
        else:
            got = run(hint)
        assert all(torch.equal(a, b) for a, b in zip(got, want)), hint
