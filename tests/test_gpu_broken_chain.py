"""The backwards whose tiles hand partial sums to each other, with waits that run out: what depends on a tile that was not waited for is NaN,
everything else is what a patient run gives, and the status says so.  No wrong number, as nobody reads the status of an ordinary call."""
import ctypes

import pytest
import torch

from test_gpu_parity import small_case

pytestmark = pytest.mark.gpu

TIMEOUT = 3


@pytest.mark.parametrize("H,D,lengths,kernels", [(8, 128, [2000, 3000, 3500], 2), (24, 64, [1500, 2100], 0), (8, 128, [2000, 1500], 2)],
                         ids=["row-tiles", "row-tiles-64", "key-tiles"])
def test_waits_that_run_out(gpu_device, H, D, lengths, kernels):
    from stickbreaking_attention import _native

    _, (q, k, v, do, drem), cu = small_case(H, D, lengths, torch.bfloat16, seed=H)
    cu = cu.to(gpu_device)
    _, _, _, carry = _native.forward(q, k, v, cu, False, max(lengths), D ** -0.5, False, want_carry=True)

    def backward(polls):
        grads = [torch.empty_like(q) for _ in range(3)]
        a = _native._base_args(q, cu, False, max(lengths), D ** -0.5, False)
        a.backward_kernels, a.carry = kernels, carry.data_ptr()
        a.q, a.k, a.v, a.d_o, a.dq, a.dk, a.dv = (_native._tensor(t, False) for t in (q, k, v, do, *grads))
        a.d_rem = _native._vector(drem, False)
        need = ctypes.c_size_t()
        assert _native.lib().sba_workspace_bytes(ctypes.byref(a), None, ctypes.byref(need), None) == 0
        ws = torch.full((need.value,), 0xFF, dtype=torch.uint8, device=q.device)
        a.workspace, a.workspace_bytes = ws.data_ptr(), need.value
        _native.ext().backward_with_polls(ctypes.addressof(a), polls)
        status = int(ws[_native.STATUS_OFFSET:_native.STATUS_OFFSET + 4].view(torch.int32).item())
        return grads, status

    whole, status = backward(0)
    assert status == 0 and all(torch.isfinite(t.float()).all() for t in whole)
    broken = 0
    for polls in (1, 1, 2, 3, 5, 8, 13, 21, 34, 55):
        got, status = backward(polls)
        nans = 0
        for n, a, b in zip(("dq", "dk", "dv"), got, whole):
            assert (torch.isnan(a) | (a == b)).all(), f"{n}, {polls} polls: a number that is neither right nor NaN"
            nans += torch.isnan(a).sum().item()
        assert (status == TIMEOUT) == (nans > 0), (polls, status, nans)
        print(f"{polls} polls: status {status}, {nans} NaN", flush=True)
        broken += status == TIMEOUT
    assert broken > 0      # (some wait ran out at all)
