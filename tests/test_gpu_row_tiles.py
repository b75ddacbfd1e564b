"""GPU tests of the backward on row tiles (csrc/sba_bwd_row.hip), which runs from 64 K rows x heads on at head_dim 64 and 128: many heads over
few rows, so that the edges of its tiles (256 rows, 32 per wave), key blocks (32) and queues are reached with an oracle in reach.

Against the float64 oracle on some heads (the bar of test_gpu_parity.py), against the dQ and dK/dV kernels on all (two orders of
summation: twice that bar), and bit for bit against itself.  Every buffer comes poisoned with NaN."""
import numpy as np
import pytest
import torch

from oracle import sb_oracle as orc
from test_gpu_backward_route import runs_on_row_tiles
from test_gpu_parity import tol_check

pytestmark = pytest.mark.gpu

CASES = [
    # label, heads, lengths, options
    ("blocks", 256, [1, 31, 32, 33, 64, 95], {}),
    ("tiles", 96, [255, 256, 257], {}),
    ("tiles-visible-diagonal", 88, [256, 257, 288, 1], dict(attend_current=True)),
    ("chain", 80, [600, 289, 33], dict(dtype=torch.float16)),
    ("long-chain", 8, [4099, 4100], {}),
    ("uneven-heads", 100, [513, 170], dict(pad=130)),
    ("odd-heads", 65, [300, 257, 224, 259], dict(token_major=True)),
    ("remainder", 72, [513, 400], dict(add_remainder=True)),
    ("remainder-rebuilt", 60, [545, 548], dict(add_remainder=True, save_carry=False, attend_current=True, dtype=torch.float16)),
    ("o-alone", 128, [512], dict(grad_rem=False, save_carry=False)),
    ("fixed", 64, [300, 300, 300, 300], dict(fixed=True)),
    ("two-launches", 64, [1100, 300] + [35] * 50, {}),      # (48 heads and 16)
    ("saturated", 80, [600, 289, 33], dict(qk_std=3.0)),
    # (head_dim 64 runs on row tiles from a mean of 512 tokens on)
    ("edges-64", 40, [255, 257, 1300, 545, 33, 900], {}),
    ("edges-visible-diagonal-64", 32, [800, 289, 511, 1025, 288], dict(attend_current=True)),
    ("odd-heads-64", 33, [545, 600, 511, 577, 560, 600, 513, 514], dict(token_major=True)),
    ("remainder-64", 40, [700, 513, 400, 600], dict(add_remainder=True)),
    ("uneven-heads-64", 36, [513, 600, 520, 545], dict(pad=130)),
    ("fixed-64", 32, [545, 545, 545, 545], dict(fixed=True)),
    ("saturated-64", 40, [600, 289, 1033], dict(qk_std=3.0)),
]


def gradients(native, mode, dev, cu, lengths, c):
    from stickbreaking_attention import sb_attn, sb_attn_varlen

    native.BACKWARD_KERNELS = mode
    q, k, v, do, drem = dev
    q, k, v = (t.detach().requires_grad_() for t in (q, k, v))
    opts = dict(attend_current=c.get("attend_current", False), add_remainder=c.get("add_remainder", False), save_carry=c.get("save_carry", True))
    if c.get("fixed"):
        def batched(t):      # (heads, tokens, ...) to (batch, heads, tokens, ...)
            return t.unflatten(1, (len(lengths), lengths[0])).transpose(0, 1)

        o, rem = sb_attn(*(batched(t) for t in (q, k, v)), **opts)
        do, drem = batched(do), batched(drem)
    else:
        o, rem = sb_attn_varlen(q, k, v, cu, max(lengths), zero_start=False, **opts)
    outs, grads = ([o, rem], [do, drem]) if c.get("grad_rem", True) else ([o], [do])
    got = torch.autograd.grad(outs, [q, k, v], grads)
    torch.cuda.synchronize()
    return got


@pytest.mark.parametrize("label,H,lengths,c", CASES, ids=[c[0] for c in CASES])
@pytest.mark.parametrize("D", [128, 64])
def test_against_oracle_and_two_kernels(gpu_device, D, label, H, lengths, c):
    from stickbreaking_attention import _native

    dtype, T, pad = c.get("dtype", torch.bfloat16), sum(lengths), c.get("pad", 0)
    # (at head_dim 64 a shorter mean runs the dQ and dK/dV kernels: the rest of the test is then of those alone)
    assert runs_on_row_tiles(H, D, lengths, c.get("fixed", False), add_remainder=c.get("add_remainder", False)) or (D == 64 and (T + pad) // len(lengths) < 512)
    g = torch.Generator().manual_seed(len(label) + H)
    q, k, v, do = (torch.randn(H, T + pad, D, generator=g) for _ in range(4))
    q, k = q * c.get("qk_std", 1.0), k * c.get("qk_std", 1.0)
    host = [t.to(dtype) for t in (q, k, v, do, torch.randn(H, T + pad, generator=g))]
    dev = [t.transpose(0, 1).contiguous().to(gpu_device).transpose(0, 1) if c.get("token_major") and t.dim() == 3 else t.to(gpu_device) for t in host]
    cu = torch.tensor(np.cumsum(lengths), dtype=torch.int32)
    saved = (_native.BACKWARD_KERNELS, _native.POISON)
    try:
        _native.POISON = True
        rows, again, two = (gradients(_native, mode, dev, cu.to(gpu_device), lengths, c) for mode in (0, 0, 1))
    finally:
        _native.BACKWARD_KERNELS, _native.POISON = saved
    heads = sorted({0, 1, H // 2, H - 1})
    hq, hk, hv, hdo, hdrem = ([t[heads][:, :T] for t in host])
    if not c.get("grad_rem", True):
        hdrem = torch.zeros_like(hdrem)
    extra = {}
    if c.get("add_remainder"):      # o + rem v: rem's gradient gains do . v, v's rem do
        hdrem = (hdrem.double() + (hdo.double() * hv.double()).sum(-1))
    ref = orc.varlen_stream(hq, hk, hv, cu, attend_current=c.get("attend_current", False), do=hdo, drem=hdrem, dtype=torch.float64)
    if c.get("add_remainder"):
        extra["dv"] = ref[1].unsqueeze(-1) * hdo.double()
    for name, a, b, w, r in zip(("dq", "dk", "dv"), rows, again, two, ref[2:]):
        assert torch.equal(a, b), f"{label}: {name} differs between two runs"
        r = r + extra.get(name, 0)
        tol_check(name, a[heads][:, :T], r, dtype, f"row tiles {label}")
        if pad:
            assert (a[:, T:] == 0).all(), f"{name}: rows no sequence covers must be zero"
        x, y = a.float(), w.float()
        assert torch.isfinite(x).all()
        ulp = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10
        excess = (x - y).abs() - 2 * torch.maximum(torch.full_like(y, 2e-2), y.abs() * ulp)
        assert excess.max().item() <= 0, f"{label}: {name} against the two kernels, {excess.max().item():.3e} beyond twice the bound"


@pytest.mark.parametrize("H,lengths", [(80, [600, 33, 289, 256, 257]), (40, [1600, 33, 900, 256, 257, 300]), (64, [1100, 300] + [35] * 50), (16, [40] * 40 + [2100, 700, 1300] + [40] * 40), (96, [255, 256, 64]), (128, [255, 256, 64])],
                         ids=["chain", "chain-64", "two-launches", "scheduler-kernel", "nothing-handed-over-two-kernels", "nothing-handed-over"])
@pytest.mark.parametrize("D", [128, 64])
def test_lengths_on_the_host_give_the_same_bits(gpu_device, D, H, lengths):
    """With the lengths on the host, what the tiles hand over is laid out by their place in the list and takes as much memory as it needs."""
    from stickbreaking_attention import _native

    g = torch.Generator().manual_seed(H)
    dev = [torch.randn(H, sum(lengths), D, generator=g).bfloat16().to(gpu_device) for _ in range(4)]
    dev.append(torch.randn(H, sum(lengths), generator=g).bfloat16().to(gpu_device))
    cu = torch.tensor(np.cumsum(lengths), dtype=torch.int32)
    saved = (_native.BACKWARD_KERNELS, _native.POISON)
    try:
        _native.POISON = True
        for got in zip(*(gradients(_native, 0, dev, t, lengths, {}) for t in (cu.to(gpu_device), cu, cu.long()))):
            assert torch.isfinite(got[0].float()).all() and torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])
    finally:
        _native.BACKWARD_KERNELS, _native.POISON = saved


@pytest.mark.parametrize("save_carry", [True, False])
@pytest.mark.parametrize("case", [(32, 128, [1300, 2100], torch.bfloat16), (64, 64, [1100], torch.bfloat16), (20, 64, [1200, 1700, 3400], torch.float16)],
                         ids=["cleared-with-the-schedule", "head-dim-64", "ranked-queues"])
def test_both_passes_in_a_graph(gpu_device, monkeypatch, case, save_carry):
    """Queues and counters are cleared anew by every replay: against the same calls made eagerly, bit for bit."""
    import test_gpu_prepared_schedule as prepared

    monkeypatch.setitem(prepared.CASES, "row tiles", case)
    prepared.test_both_passes_in_a_graph(gpu_device, monkeypatch, "row tiles", save_carry)
