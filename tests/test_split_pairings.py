"""The forward, dQ and dK/dV of a call each have a line of their own below which they split keys or rows over the waves: every pairing of a split with
an unsplit kernel reads only slots of the product and prefix planes that were written (host model in test_carry_slots_model.py)."""
import pytest

from test_carry_slots_model import bits, cdiv, dkv_reads, dq_carry_reads, dq_prefix_writes, forward_writes, slot

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


@pytest.mark.parametrize("keys,rows,variant", [(64, 64, "producer64"), (128, 32, "pipelined128")])
def test_sweeps_that_begin_with_the_tiles_own_rows(keys, rows, variant):
    """With the remainder in dV a tile's sweep begins with its own rows also where they do not attend to themselves: a last key that no row sees
    then gets a step.  That step fetches slots of the sequence only, and puts none to use that another sweep would not."""
    for L in [*range(1, 200), 257, 321, 385, 512, 513, 640, 641, 673]:
        used, m = (set(), set()), cdiv(L, 128)
        for j0 in range(0, L, keys):
            for w_first in range(j0 // rows * rows, rows * cdiv(L, rows), 32):
                for jb in range(j0, j0 + keys, 32):
                    fetched = {slot(jb // 32, row, m) for row in range(w_first, w_first + 32)}      # (asserts the range)
                    if w_first < L and jb <= min(w_first + 31, L - 1) - 1:
                        for u in used:
                            u.update(fetched)
        assert used == dkv_reads(L, 0, variant), L
