"""The fp32 backward whose streamed operands a kernel in front has split and laid out (sequences of 1024 tokens or more on average): against the
float64 oracle, and the same bits as where the workspace has no room for that, of which it then takes no more than it is left."""
import pytest
import torch

from oracle import sb_oracle as orc
from stickbreaking_attention import _native, sb_attn, sb_attn_varlen
from test_gpu_parity import NAMES, run_varlen, small_case

pytestmark = pytest.mark.gpu


def backward_bytes(D, H, lengths, planes=True):
    a = _native.SbaArgs()
    a.dtype, a.head_dim, a.num_heads, a.num_seqs = _native.SBA_F32, D, H, len(lengths)
    a.total_tokens, a.max_seqlen, a.cu_seqlens = sum(lengths), max(lengths), 256      # (not read: packed sequences)
    of_planes = (sum(lengths) // 32 + len(lengths) + 1) * H * 32 * 24 * (-(-D // 32) * 32)
    return _native._workspace_bytes(a)[1] - (0 if planes else of_planes)


@pytest.mark.parametrize("lengths,attend_current,add_remainder,token_major", [([1056, 1153, 994], False, False, False),
                                                                             ([1, 2271, 801], True, True, True)])
@pytest.mark.parametrize("D", [7, 32, 50, 64, 96, 128])
def test_against_oracle_and_without_room(gpu_device, D, lengths, attend_current, add_remainder, token_major):
    H = 3      # (9609 and 9219 rows x heads: products of triples)
    (q, k, v, do, drem), dev, cu = small_case(H, D, lengths, torch.float32, seed=D)
    if token_major:
        dev = [t.transpose(0, 1).contiguous().transpose(0, 1) for t in dev]

    def run():
        return run_varlen(dev[0], dev[1], dev[2], cu.to(gpu_device), lengths, False, attend_current, dev[3], dev[4], add_remainder=add_remainder)

    outs = run()
    whole, pieces = backward_bytes(D, H, lengths), sum(lengths) // 32 + len(lengths) + 1
    assert whole > 4 * pieces * H * 32 * 6 * D      # the planes are part of what is asked for
    _native.set_backward_workspace_limit(whole - 1)
    try:
        without = run()
    finally:
        _native.set_backward_workspace_limit(None)
    d = [t.double() for t in (q, k, v, do, drem)]
    if add_remainder:
        d[4] = orc.remainder_drem(d[3], d[4], d[2])
    ref = orc.varlen_stream(d[0], d[1], d[2], cu, attend_current=attend_current, do=d[3], drem=d[4], dtype=torch.float64)
    if add_remainder:
        ref = orc.with_remainder(ref, d[2], d[3])
    for n, a, b, r in zip(NAMES, outs, without, ref):
        rel = (a.detach().double().cpu() - r).norm() / r.norm()
        print(f"D={D} {n}: relative error {rel.item():.2e}", flush=True)
        assert rel < 1e-5, f"{n}: {rel.item():.2e}"      # (fp32 sums over up to 2271 terms: sqrt(2271) 2^-24 = 3e-6)
        assert torch.equal(a, b), f"{n}: laid out and not differ"


@pytest.mark.parametrize("D", [50, 128])
@pytest.mark.parametrize("L", [1024, 1057])
def test_of_one_length(gpu_device, L, D):
    B, H = 3, 3
    g = torch.Generator().manual_seed(L + D)
    host = [torch.randn(B, H, L, D, generator=g) for _ in range(4)] + [torch.randn(B, H, L, generator=g)]
    q, k, v, do, drem = (t.to(gpu_device) for t in host)
    for t in (q, k, v):
        t.requires_grad_()

    def run():
        o, rem = sb_attn(q, k, v)
        return (o, rem, *torch.autograd.grad([o, rem], [q, k, v], [do, drem]))

    outs = run()
    a = _native.SbaArgs()
    a.dtype, a.head_dim, a.num_heads, a.num_seqs, a.total_tokens, a.max_seqlen = _native.SBA_F32, D, H, B, L, L
    _native.set_backward_workspace_limit(_native._workspace_bytes(a)[1] - 1)
    try:
        without = run()
    finally:
        _native.set_backward_workspace_limit(None)
    cu = torch.tensor([L], dtype=torch.int32)
    for b in range(B):
        d = [t[b].double() for t in host]
        ref = orc.varlen_stream(*d[:3], cu, do=d[3], drem=d[4], dtype=torch.float64)
        for n, x, r in zip(NAMES, outs, ref):
            assert (x[b].detach().double().cpu() - r).norm() / r.norm() < 1e-5, n      # (as above)
    for n, x, y in zip(NAMES, outs, without):
        assert torch.equal(x, y), f"{n}: laid out and not differ"


def long_case(device, H, D, lengths):
    g = torch.Generator(device=device).manual_seed(D)
    q, k, v, do = (torch.randn(H, sum(lengths), D, generator=g, device=device) for _ in range(4))
    for t in (q, k, v):
        t.requires_grad_()
    o, rem = sb_attn_varlen(q, k, v, torch.tensor(lengths).cumsum(0).int().to(device), max(lengths), zero_start=False)
    return lambda: torch.autograd.grad(o, [q, k, v], do, retain_graph=True)


def peak_of(backward, results):
    """What a backward takes besides its results."""
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    grads = backward()
    torch.cuda.synchronize()
    return grads, torch.cuda.max_memory_allocated() - before - results


def test_groups_of_heads_with_planes(gpu_device):
    """A workspace that holds three of five heads with their planes, and not all of them without."""
    H, D, lengths = 5, 32, [20001, 479]
    backward = long_case(gpu_device, H, D, lengths)
    whole = backward()
    limit = backward_bytes(D, H, lengths, planes=False) - 1
    assert backward_bytes(D, 3, lengths) <= limit and backward_bytes(D, 3, lengths) > backward_bytes(D, 3, lengths, planes=False)
    _native.set_backward_workspace_limit(limit)
    try:
        in_groups = backward()
    finally:
        _native.set_backward_workspace_limit(None)
    for n, x, y in zip(NAMES[2:], whole, in_groups):
        assert torch.equal(x, y), n


@pytest.mark.parametrize("host_layer", [True, False])
def test_a_limit_below_what_one_head_asks_for_is_kept(gpu_device, monkeypatch, host_layer):
    if not host_layer:
        monkeypatch.setattr(_native, "use_ext", lambda: False)
    H, D, lengths = 2, 128, [4096]
    backward = long_case(gpu_device, H, D, lengths)
    whole = backward()
    limit = backward_bytes(D, 1, lengths, planes=False) + (1 << 20)
    assert limit + (8 << 20) < backward_bytes(D, 1, lengths)
    _native.set_backward_workspace_limit(limit)
    try:
        grads, peak = peak_of(backward, 3 * H * sum(lengths) * D * 4)
    finally:
        _native.set_backward_workspace_limit(None)
    slack = 64 << 10      # (the rows' zero gradients of rem, blocks rounded up)
    assert peak <= limit + slack
    for n, x, y in zip(NAMES[2:], whole, grads):
        assert torch.equal(x, y), n


@pytest.mark.parametrize("host_layer", [True, False])
@pytest.mark.parametrize("H,lengths", [(1, [24576]), (4, [8192, 8192])])
def test_little_memory_left(gpu_device, monkeypatch, H, lengths, host_layer):
    """Room for all heads, one or several, without planes only: they run in one pass."""
    if not host_layer:
        monkeypatch.setattr(_native, "use_ext", lambda: False)
    D, device = 128, torch.cuda.current_device()
    whole = [t.cpu() for t in long_case(gpu_device, H, D, lengths)()]
    backward = long_case(gpu_device, H, D, lengths)
    results = 3 * H * sum(lengths) * D * 4
    least, most = backward_bytes(D, H, lengths, planes=False), backward_bytes(D, H, lengths)
    left = least + (6 << 20)
    assert left + (32 << 20) < most
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(device).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + results + left) / total)
    try:
        for scheduled in ("by the forward", "by the backward"):
            grads, peak = peak_of(backward, results)
            assert 0.9 * least < peak < most, scheduled      # (not a group of heads)
            for n, x, y in zip(NAMES[2:], whole, grads):
                assert torch.equal(x, y.cpu()), f"{n}, scheduled {scheduled}"
            del grads, y
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
