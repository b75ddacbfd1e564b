"""A max_seqlens of up to 64 that a sequence exceeds.  A backward for sequences of up to 64 tokens alone would leave that one's gradients unwritten, so
the call is void in both passes, also where the carry buffer would hold the products; a forward that no backward follows stands."""
import numpy as np
import pytest
import torch

from oracle import sb_oracle as orc
from stickbreaking_attention import _native, sb_attn_varlen
from test_gpu_device_void import CARRY_TOO_SMALL, _backward, _forward, _inputs
from test_gpu_parity import NAMES, tol_check

pytestmark = pytest.mark.gpu

FEW, MANY = [100, 65, 300, 20], [20] * 40 + [100] + [20] * 40      # scheduled by the forward, by the scheduler kernel


@pytest.mark.parametrize("lengths", [FEW, MANY], ids=["few", "many"])
@pytest.mark.parametrize("H,D,kernels", [(2, 64, 0), (8, 128, 0), (12, 50, 1), (8, 128, 2)])
def test_void_in_both_passes(gpu_device, H, D, kernels, lengths):
    q, k, v = _inputs(H, sum(lengths), D, torch.bfloat16, gpu_device)
    cu = torch.tensor(np.cumsum(lengths), dtype=torch.int32, device=gpu_device)
    for most, expected in ((64, CARRY_TOO_SMALL), (max(lengths), 0)):
        for kept in (True, False):
            ret, status, outs, carry = _forward(_native, q, k, v, cu, most, 0, want_carry=kept, recompute=not kept)
            assert ret == 0 and status == expected
            assert all(bool((t == 0).all()) == bool(expected) for t in outs)
            ret, status, grads = _backward(_native, q, k, v, cu, most, 0, carry if kept else None, kernels)
            assert ret == 0 and status == expected
            assert all(bool((t == 0).all()) == bool(expected) and not (t == 7).all() for t in grads)


@pytest.mark.parametrize("lengths", [FEW, MANY], ids=["few", "many"])
@pytest.mark.parametrize("save_carry", [True, False])
def test_operators(gpu_device, lengths, save_carry):
    assert _native.DEBUG_CHECK
    q, k, v = _inputs(2, sum(lengths), 64, torch.bfloat16, gpu_device)
    cu = torch.tensor(np.cumsum(lengths), dtype=torch.int32, device=gpu_device)
    with torch.no_grad():
        alone = sb_attn_varlen(q, k, v, cu, 64, zero_start=False)
    ref = orc.varlen_stream(*(t.double().cpu() for t in (q, k, v)), cu.cpu(), dtype=torch.float64)
    for n, a, b in zip(NAMES, alone, ref):
        tol_check(n, a, b, torch.bfloat16, "forward alone")
    for limit in (None, 1):
        _native.set_backward_workspace_limit(limit)
        try:
            with pytest.raises(ValueError, match="max_seqlens understated"):
                sb_attn_varlen(q.requires_grad_(), k, v, cu, 64, zero_start=False, save_carry=save_carry)
        finally:
            _native.set_backward_workspace_limit(None)


def test_fixed_length_mode_goes_by_the_shape(gpu_device, monkeypatch):
    B, H, L, D = 2, 8, 100, 128
    g = torch.Generator().manual_seed(5)
    host = [torch.randn(B, H, L, D, generator=g).bfloat16() for _ in range(4)] + [torch.randn(B, H, L, generator=g).bfloat16()]
    q, k, v, do, drem = (t.to(gpu_device) for t in host)
    base_args = _native._base_args

    def understated(*args, **kw):
        a = base_args(*args, **kw)
        a.max_seqlen = 64
        return a

    monkeypatch.setattr(_native, "_base_args", understated)
    o, rem, _, carry = _native.forward(q, k, v, None, False, L, D ** -0.5, False, True)
    got = (o, rem, *_native.backward(do, drem, q, k, v, carry, None, False, L, D ** -0.5, False))
    cu = torch.tensor([L], dtype=torch.int32)
    for b in range(B):
        d = [t[b].double() for t in host]
        ref = orc.varlen_stream(*d[:3], cu, do=d[3], drem=d[4], dtype=torch.float64)
        for n, x, r in zip(NAMES, got, ref):
            tol_check(n, x[b], r, torch.bfloat16, f"sequence {b}")
