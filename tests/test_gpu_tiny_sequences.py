"""The backward of sequences of up to 64 tokens (csrc/sba_bwd_tiny.hip), alone and beside longer ones: lengths around its 32-row blocks, empty sequences,
rows no sequence covers, every head_dim class, with and without the remainder, recorded and rebuilt products; against the float64 oracle."""
import numpy as np
import pytest
import torch

from oracle import sb_oracle as orc
from stickbreaking_attention import _native, sb_attn, sb_attn_varlen
from test_gpu_parity import NAMES, tol_check

pytestmark = pytest.mark.gpu


def check(device, H, D, lengths, dtype=torch.bfloat16, pad=0, fixed=False, token_major=False, attend_current=False, add_remainder=False, save_carry=True, host_cu=False):
    T = sum(lengths)
    g = torch.Generator().manual_seed(T * H + D)
    host = [torch.randn(H, T + pad, D, generator=g).to(dtype) for _ in range(4)] + [torch.randn(H, T + pad, generator=g).to(dtype)]
    dev = [t.to(device) for t in host]
    if token_major:
        dev = [t.transpose(0, 1).contiguous().transpose(0, 1) for t in dev]
    q, k, v = (t.detach().requires_grad_() for t in dev[:3])
    options = dict(attend_current=attend_current, add_remainder=add_remainder, save_carry=save_carry)
    saved = _native.POISON
    try:
        _native.POISON = True
        if fixed:
            def batched(t):
                return t.unflatten(1, (len(lengths), lengths[0])).transpose(0, 1)

            o, rem = sb_attn(batched(q), batched(k), batched(v), **options)
            got = [t.transpose(0, 1).flatten(1, 2) for t in (o, rem)] + list(torch.autograd.grad([o, rem], [q, k, v], [batched(dev[3]), batched(dev[4])]))
        else:
            cu = torch.tensor(np.cumsum(lengths), dtype=torch.int32)
            o, rem = sb_attn_varlen(q, k, v, cu if host_cu else cu.to(device), max(lengths), zero_start=False, **options)
            got = [o, rem, *torch.autograd.grad([o, rem], [q, k, v], dev[3:])]
    finally:
        _native.POISON = saved
    heads = sorted({0, H - 1})
    d = [t[heads, :T].double() for t in host]
    if add_remainder:
        d[4] = orc.remainder_drem(d[3], d[4], d[2])
    cu = torch.tensor(np.cumsum(lengths), dtype=torch.int32)
    ref = orc.varlen_stream(d[0], d[1], d[2], cu, attend_current=attend_current, do=d[3], drem=d[4], dtype=torch.float64)
    if add_remainder:
        ref = orc.with_remainder(ref, d[2], d[3])
    for n, a, b in zip(NAMES, got, ref):
        tol_check(n, a[heads, :T], b, dtype, f"H={H} D={D}")
        assert (a[:, T:] == 0).all(), f"{n}: rows no sequence covers must be zero"


EDGES = [64, 1, 31, 32, 33, 2, 63, 16, 0, 48, 34, 64]


@pytest.mark.parametrize("attend_current,add_remainder,save_carry", [(False, False, True), (True, True, False), (False, True, True), (True, False, True)])
@pytest.mark.parametrize("H,D", [(3, 8), (2, 50), (8, 64), (5, 100), (8, 128)])
def test_alone(gpu_device, H, D, attend_current, add_remainder, save_carry):
    check(gpu_device, H, D, EDGES, pad=40, attend_current=attend_current, add_remainder=add_remainder, save_carry=save_carry)


@pytest.mark.parametrize("D", [64, 72, 128])
@pytest.mark.parametrize("L", [1, 32, 33, 64])
def test_of_one_length(gpu_device, L, D):
    check(gpu_device, 4, D, [L] * 5, fixed=True)
    check(gpu_device, 4, D, [L] * 5, dtype=torch.float16, token_major=True)


@pytest.mark.parametrize("host_cu", [False, True])
@pytest.mark.parametrize("H,D,longer", [(16, 50, [300, 65, 700]), (32, 64, [128, 129]), (32, 128, [300, 65, 1000, 257]), (16, 80, [900]), (32, 128, [4000]), (32, 64, [16000])])
def test_beside_longer_ones(gpu_device, H, D, longer, host_cu):
    """More than 64 sequences (the scheduler kernel lists them) and, of one case, up to 64 (the forward does)."""
    rng = np.random.default_rng(D)
    for count in (61, 300):
        lengths = [int(x) for x in rng.integers(0, 65, count)]
        for n in longer:
            lengths.insert(int(rng.integers(0, len(lengths))), n)
        if sum(lengths) < 128 * len(lengths):
            check(gpu_device, H, D, lengths, pad=7, host_cu=host_cu)
