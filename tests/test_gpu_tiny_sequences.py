"""The backward of sequences of up to 64 tokens (csrc/sba_bwd_tiny.hip), alone and beside longer ones: lengths around its 32-row blocks, empty sequences,
rows no sequence covers, every head_dim class, with and without the remainder, recorded and rebuilt products; against the float64 oracle."""
import ctypes

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


def form_and_kernels(H, D, lengths, dtype=torch.bfloat16, add_remainder=False):
    a = _native.SbaArgs()
    a.dtype, a.head_dim, a.num_heads, a.num_seqs = _native.SBA_BF16 if dtype == torch.bfloat16 else _native.SBA_F16, D, H, len(lengths)
    a.total_tokens, a.max_seqlen, a.add_remainder, a.cu_seqlens = sum(lengths), max(lengths), int(add_remainder), 256      # (not read: packed sequences)
    a.workspace_bytes = 1 << 40
    return _native.ext().backward_route(ctypes.addressof(a))[0], _native.lib().sba_bwd_kernels(ctypes.byref(a))


def among(count, longer):
    rng = np.random.default_rng(count)
    lengths = [int(x) for x in rng.integers(0, 65, count)]
    for n in longer:
        lengths.insert(int(rng.integers(0, len(lengths))), n)
    return lengths


LONG = [300, 65, 1000, 257]
BESIDE = [(16, 50, [300, 65, 700]), (32, 64, [128, 129]), (32, 128, LONG), (16, 80, [900]), (32, 128, [4000]), (32, 64, [16000])]


@pytest.mark.parametrize("host_cu", [False, True])
@pytest.mark.parametrize("H,D,longer,count", [(*c, 300) for c in BESIDE] + [(*c, 61) for c in BESIDE[:-1]])
def test_beside_longer_ones(gpu_device, H, D, longer, count, host_cu):
    """Taken apart in batches of more than 64 sequences; up to 64 the longer ones' kernels take them too."""
    lengths = among(count, longer)
    form, kernels = form_and_kernels(H, D, lengths)
    assert kernels == (1 if form == _native.KEY_TILES else 2) + (len(lengths) > 64)
    check(gpu_device, H, D, lengths, pad=7, host_cu=host_cu)


KEYS = [1 + i % 15 for i in range(70)] + [65, 100, 35]


@pytest.mark.parametrize("H,D,lengths,options,form", [
    (8, 128, KEYS * 2, {}, _native.KEY_TILES), (8, 128, KEYS * 2, dict(dtype=torch.float16, save_carry=False), _native.KEY_TILES),
    (8, 128, KEYS * 2, dict(attend_current=True, token_major=True), _native.KEY_TILES),
    (32, 128, among(300, LONG), dict(dtype=torch.float16, add_remainder=True), _native.ROW_TILES),
    (32, 128, among(300, LONG), dict(attend_current=True, save_carry=False), _native.ROW_TILES),
    (16, 64, among(300, LONG), dict(add_remainder=True, save_carry=False), _native.TWO_KERNELS),
    (5, 80, among(300, LONG), dict(dtype=torch.float16, attend_current=True, add_remainder=True), _native.TWO_KERNELS)])
def test_beside_each_form_with_each_option(gpu_device, H, D, lengths, options, form):
    got = form_and_kernels(H, D, lengths, options.get("dtype", torch.bfloat16), options.get("add_remainder", False))
    assert got == (form, 2 if form == _native.KEY_TILES else 3)      # one of them the tiny ones'
    check(gpu_device, H, D, lengths, pad=7, **options)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("longest", [None, 4096])
def test_none_longer_after_all(gpu_device, D, longest):
    """Lengths on the device only and a bound far above them: the kernels of longer sequences run on no tile, and clear the rows of no sequence."""
    lengths = among(300, [])
    H, T = 16, sum(lengths)
    g = torch.Generator().manual_seed(D)
    host = [torch.randn(H, T + 300, D, generator=g).bfloat16() for _ in range(4)] + [torch.randn(H, T + 300, generator=g).bfloat16()]
    q, k, v, do, drem = (t.to(gpu_device) for t in host)
    for t in (q, k, v):
        t.requires_grad_()
    cu = torch.tensor(np.cumsum(lengths), dtype=torch.int32)
    o, rem = sb_attn_varlen(q, k, v, cu.to(gpu_device), longest, zero_start=False)
    got = (o, rem, *torch.autograd.grad([o, rem], [q, k, v], [do, drem]))
    d = [t[:1, :T].double() for t in host]
    for n, a, b in zip(NAMES, got, orc.varlen_stream(*d[:3], cu, do=d[3], drem=d[4], dtype=torch.float64)):
        tol_check(n, a[:1, :T], b, torch.bfloat16, f"D={D}")
        assert (a[:, T:] == 0).all(), f"{n}: rows no sequence covers must be zero"


@pytest.mark.parametrize("H,D,longer", [(16, 64, LONG), (32, 128, LONG), (32, 128, [])])
def test_heads_in_groups(gpu_device, monkeypatch, H, D, longer):
    """Under a workspace limit the groups take the tiny sequences as one pass over all heads would: the same bits of their gradients."""
    monkeypatch.setattr(_native, "BACKWARD_KERNELS", 0)      # (2 takes none apart)
    lengths = among(300, longer)
    g = torch.Generator(device=gpu_device).manual_seed(D)
    q, k, v, do = (torch.randn(H, sum(lengths), D, generator=g, device=gpu_device).bfloat16() for _ in range(4))
    for t in (q, k, v):
        t.requires_grad_()
    cu = torch.tensor(np.cumsum(lengths), dtype=torch.int32, device=gpu_device)
    tiny = torch.cat([torch.arange(e - n, e) for n, e in zip(lengths, np.cumsum(lengths)) if n <= 64]).to(gpu_device)
    o, _ = sb_attn_varlen(q, k, v, cu, max(lengths), zero_start=False)
    whole = torch.autograd.grad(o, [q, k, v], do)
    _native.set_backward_workspace_limit(1)      # (a head at a time)
    try:
        o, _ = sb_attn_varlen(q, k, v, cu, max(lengths), zero_start=False)
        one_by_one = torch.autograd.grad(o, [q, k, v], do)
    finally:
        _native.set_backward_workspace_limit(None)
    for n, a, b in zip(NAMES[2:], whole, one_by_one):
        assert torch.equal(a[:, tiny], b[:, tiny]), n
        assert (a.float() - b.float()).norm() <= 1e-2 * a.float().norm(), n      # (the longer ones on other kernels: a rounding to 8 bits of P and dZ)
