"""Batches whose tiles the forward's workgroups list themselves, a sequence per lane: counts around the rows of 16 lanes that the sums are formed over
and up to the last lane, lengths on both sides of the four query tiles a lane lists itself, empty sequences.  Against the float64 oracle."""
import numpy as np
import pytest
import torch

from oracle import sb_oracle as orc
from stickbreaking_attention import sb_attn_varlen
from test_gpu_parity import NAMES, tol_check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,D", [(1, 64), (3, 50), (8, 128)])
@pytest.mark.parametrize("count", [2, 15, 16, 17, 33, 49, 63, 64])
def test_sequences_in_lanes(gpu_device, count, H, D):
    rng = np.random.default_rng(count)
    lengths = [int(x) for x in rng.integers(0, 150, count)]
    for i, n in zip(rng.choice(count, min(count, 6), replace=False), [900, 511, 513, 0, 512, 640]):
        lengths[i] = n
    T = sum(lengths)
    g = torch.Generator().manual_seed(count)
    host = [torch.randn(H, T, D, generator=g).bfloat16() for _ in range(4)] + [torch.randn(H, T, generator=g).bfloat16()]
    q, k, v, do, drem = (t.to(gpu_device) for t in host)
    for t in (q, k, v):
        t.requires_grad_()
    cu = torch.tensor(np.cumsum(lengths), dtype=torch.int32)
    o, rem = sb_attn_varlen(q, k, v, cu.to(gpu_device), max(lengths), zero_start=False)
    got = (o, rem, *torch.autograd.grad([o, rem], [q, k, v], [do, drem]))
    d = [t[:1].double() for t in host]
    ref = orc.varlen_stream(d[0], d[1], d[2], cu, do=d[3], drem=d[4], dtype=torch.float64)
    for n, a, b in zip(NAMES, got, ref):
        tol_check(n, a[:1], b, torch.bfloat16, f"{count} sequences")
