"""The fp32 backward whose streamed operands a kernel in front has split and laid out (sequences of 1024 tokens or more on average): against the
float64 oracle, and the same bits as where the workspace has no room for that."""
import pytest
import torch

from oracle import sb_oracle as orc
from stickbreaking_attention import _native
from test_gpu_parity import NAMES, run_varlen, small_case

pytestmark = pytest.mark.gpu


def backward_bytes(D, H, lengths):
    a = _native.SbaArgs()
    a.dtype, a.head_dim, a.num_heads, a.num_seqs = _native.SBA_F32, D, H, len(lengths)
    a.total_tokens, a.max_seqlen, a.cu_seqlens = sum(lengths), max(lengths), 256      # (not read: packed sequences)
    return _native._workspace_bytes(a)[1]


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
