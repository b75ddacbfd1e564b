"""The forward, dQ and dK/dV of a call each have a line of their own below which they split keys or rows over the waves: every pairing of a split with
an unsplit kernel reads only slots of the product and prefix planes that were written (host model in test_carry_slots_model.py)."""
import pytest

from test_carry_slots_model import bits, dkv_reads, dq_carry_reads, dq_prefix_writes, forward_writes

PAIRINGS = [(f, dq, d) for f in (32, "split") for dq in (32, "split") for d in ("producer64", "pipelined128", "chained")] + \
           [(f, dq, d) for f in (64, "split") for dq in (32, "split") for d in ("wave", "split")]


@pytest.mark.parametrize("fwd_kt,dq_kt,dkv", PAIRINGS)
@pytest.mark.parametrize("ac", [0, 1])
def test_every_slot_read_was_written(fwd_kt, dq_kt, dkv, ac):
    for L in [*range(1, 200), 255, 256, 257, 289, 385, 511, 512, 513, 640, 641, 673]:
        written_carry, written_prefix = bits(forward_writes, L, ac, fwd_kt), bits(dq_prefix_writes, L, ac, dq_kt)
        carry, prefix = bits(dkv_reads, L, ac, dkv)
        assert (bits(dq_carry_reads, L, ac, dq_kt) | carry) & ~written_carry == 0, L
        assert prefix & ~written_prefix == 0, L
