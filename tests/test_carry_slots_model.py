"""Host model of which carry / prefix slots each kernel variant writes and which it reads.

The forward records, per (row, 32-key sub-tile), the product of (1 - sigma) above the sub-tile (`carry`), the dQ
kernel records the prefix sum of g below it (`prefix`), and the dK/dV kernels start their scans from both.  The
buffers come from the allocator uninitialised, so every slot a dK/dV or dQ variant reads with its math enabled must
have been written by whichever forward / dQ variant ran before it -- for every sequence length, for both
`attend_current` settings and for every pairing of variants the launcher can produce (each pass chooses by how the rows
of its own tensors can be read; the 16-bit kernels of one call agree on whether the call is small).  The index arithmetic
below restates, variant by variant, the loop bounds and skip tests of csrc/sba_fwd.hip, sba_bwd_dq.hip, sba_bwd_dkv.hip,
sba_split.hip, sba_bwd_chain.hip and sba_f32.hip; the GPU suite checks the same property on the device by poisoning the
buffers with NaN.

Rows of a 32-row block that lies beyond the sequence's end as a whole do not count as read: where a kernel computes them at
all, a row's values stay in its own lanes and are dropped at the end.
"""
import functools

import numpy as np
import pytest

BQ = 128


def cdiv(a, b):
    return -(-a // b)


def carry_offset(u, m):
    q, r = u >> 2, u & 3
    return u * (m * 128) - 128 * (2 * q * (q - 1) + r * q)


def slot(u, row, m):
    """Flat slot of (sub-tile u, row) in a sequence of m query tiles, with the range checks the layout implies."""
    assert 0 <= u < 4 * m and BQ * (u >> 2) <= row < BQ * m, (u, row, m)
    s = carry_offset(u, m) + (row - BQ * (u >> 2))
    assert 0 <= s < 256 * m * (m + 1)
    return s


def tile_key_steps(L, ac, qt, kt):
    last_row = min(BQ * qt + BQ, L) - 1
    last_key = last_row - 1 + ac
    return 0 if last_key < 0 else last_key // kt + 1


def split_blocks(L, ac, step):
    """The 32-row blocks of a sequence, each swept by itself in steps of `step` keys: (first row, steps, last visible key)."""
    for q0 in range(0, L, 32):
        last_key = min(q0 + 32, L) - 2 + ac
        yield q0, (0 if last_key < 0 else last_key // step + 1), last_key


def forward_writes(L, ac, kt):
    m, out = cdiv(L, BQ), set()
    if kt in ("split", "f32"):
        for q0, n, _ in split_blocks(L, ac, 128 if kt == "split" else 32):
            for u in range(4 * n if kt == "split" else n):      # split: every sub-tile of a step, whichever wave's it is
                for row in range(q0, q0 + 32):
                    out.add(slot(u, row, m))
        return out
    for qt in range(m):
        n = tile_key_steps(L, ac, qt, kt)
        subs = list(range(n)) if kt == 32 else list(range(2 * n))
        if kt == 32 and n % 2 == 1:
            subs.append(n)                      # the product above the upper half of the last 64-key tile
        for u in subs:
            for row in range(BQ * qt, BQ * qt + BQ):
                out.add(slot(u, row, m))
    return out


def dq_prefix_writes(L, ac, kt):
    m, out = cdiv(L, BQ), set()
    if kt in ("split", "f32"):
        for q0, _, last_key in split_blocks(L, ac, 128):
            for u in range(0, last_key // 32 + 1):
                for row in range(q0, q0 + 32):
                    out.add(slot(u, row, m))
        return out
    for qt in range(m):
        n = tile_key_steps(L, ac, qt, kt)
        for u in (range(n) if kt == 32 else range(2 * n)):
            for row in range(BQ * qt, BQ * qt + BQ):
                out.add(slot(u, row, m))
    return out


def dq_carry_reads(L, ac, kt):
    if kt in ("split", "f32"):
        return dq_prefix_writes(L, ac, kt)      # one product in, one prefix sum out, for every sub-tile a wave works on
    m, out = cdiv(L, BQ), set()
    for qt in range(m):
        for jt in range(tile_key_steps(L, ac, qt, kt)):
            u = jt if kt == 32 else 2 * jt + 1
            for row in range(BQ * qt, min(BQ * qt + BQ, 32 * cdiv(L, 32))):
                out.add(slot(u, row, m))
    return out


def dkv_reads(L, ac, variant, rows_beyond_end_count=False):
    """(carry slots, prefix slots) read with the element-wise math enabled."""
    m = cdiv(L, BQ)
    carry, prefix = set(), set()
    last = (lambda w_last: w_last) if rows_beyond_end_count else (lambda w_last: min(w_last, L - 1))
    if variant == "f32":                    # 32 keys, row blocks from the keys' own on, none skipped
        for k0 in range(0, L, 32):
            for b in range(k0 // 32, cdiv(L, 32) if k0 + 1 - ac < L else 0):
                for row in range(32 * b, 32 * b + 32):
                    carry.add(slot(k0 // 32, row, m))
                    prefix.add(slot(k0 // 32, row, m))
    elif variant in ("split", "wave"):      # 32 keys per workgroup, rows in steps of 128; 32 keys per wave of a 128-key tile
        for k0 in range(0, L, 32):
            first_row = (k0 if variant == "split" else k0 // 128 * 128) + 1 - ac
            step = 128 if variant == "split" else 32
            for t in range(first_row // step, cdiv(L, step)) if first_row < L else ():
                for w_first in range(step * t, step * t + step, 32):
                    if w_first >= L or k0 > last(w_first + 31) - 1 + ac:
                        continue
                    for row in range(w_first, w_first + 32):
                        carry.add(slot(k0 // 32, row, m))
                        prefix.add(slot(k0 // 32, row, m))
    elif variant in ("pipelined128", "chained"):      # 128-key tiles, steps of 32 rows, producer g = sub-tile g
        for j0 in range(0, L, 128):
            first_row = j0 + 1 - ac
            if first_row >= L:
                continue
            row_begin = (first_row // 32) * 32
            for t in range(cdiv(L - row_begin, 32)):
                q0 = row_begin + 32 * t
                for g in range(4):
                    jb = j0 + 32 * g
                    if jb > last(q0 + 31) - 1 + ac or jb >= L:
                        continue
                    for row in range(q0, q0 + 32):
                        carry.add(slot(j0 // 32 + g, row, m))
                        if variant != "chained":      # (its prefix sums are handed from tile to tile)
                            prefix.add(slot(j0 // 32 + g, row, m))
    elif variant == "producer64":          # 64-key tiles, steps of 64 rows, producer (rg, group)
        for j0 in range(0, L, 64):
            first_row = j0 + 1 - ac
            if first_row >= L:
                continue
            row_begin = (first_row // 64) * 64
            for t in range(cdiv(L - row_begin, 64)):
                for rg in range(2):
                    w_first = row_begin + 64 * t + 32 * rg
                    for group in range(2):
                        jb = j0 + 32 * group
                        if w_first >= L or jb > last(w_first + 31) - 1 + ac or jb >= L:
                            continue
                        for row in range(w_first, w_first + 32):
                            carry.add(slot(j0 // 32 + group, row, m))
                            prefix.add(slot(j0 // 32 + group, row, m))
    else:                                   # generic: 64-key tiles, 128-row query tiles, a wave per 32 rows
        for j0 in range(0, L, 64):
            first_row = j0 + 1 - ac
            if first_row >= L:
                continue
            for qt in range(first_row // BQ, m):
                for w in range(4):
                    w_first = BQ * qt + 32 * w
                    if w_first >= L or j0 > last(w_first + 31) - 1 + ac:
                        continue
                    for row in range(w_first, w_first + 32):
                        carry.add(slot(j0 // 32 + 1, row, m))
                        prefix.add(slot(j0 // 32, row, m))
    return carry, prefix


# (forward, dQ, dK/dV): what the launchers can pair up.  A pass reads its rows aligned or padded (forward: 32-key steps at
# head_dims above 64, 64-key steps below; dQ: 32), or element by element (64-key steps); a call is small for the forward and dQ
# ("split"), for dK/dV ("split" up to head_dim 64, "producer64" above), for both, or for neither.
ABOVE_64 = [(f, 32, d) for f in (32, 64) for d in ("producer64", "pipelined128", "chained")] + \
           [("split", "split", d) for d in ("producer64", "chained", "pipelined128")] + [(64, "split", "producer64")]
UP_TO_64 = [(64, 32, "wave"), (64, 32, "split"), ("split", "split", "split"), (64, "split", "split")]
BY_ELEMENT = [(f, 64, "generic") for f in (32, 64, "split")]
PAIRINGS = ABOVE_64 + UP_TO_64 + BY_ELEMENT + [("f32", "f32", "f32")]


@functools.lru_cache(maxsize=None)
def bits(fn, *args):
    """The set(s) of slots `fn` returns, as integers with a bit per slot (kept: every variant is in several pairings)."""
    def one(slots):
        flags = np.zeros(max(slots, default=0) + 1, dtype=bool)
        flags[list(slots)] = True
        return int.from_bytes(np.packbits(flags, bitorder="little").tobytes(), "little")

    got = fn(*args)
    return tuple(one(x) for x in got) if isinstance(got, tuple) else one(got)


@pytest.mark.parametrize("fwd_kt,dq_kt,dkv", PAIRINGS)
@pytest.mark.parametrize("ac", [0, 1])
def test_every_slot_read_was_written(fwd_kt, dq_kt, dkv, ac):
    lengths = list(range(1, 420)) + [511, 512, 513, 640, 641, 673, 705, 1000]
    for L in lengths:
        written_carry = bits(forward_writes, L, ac, fwd_kt)
        written_prefix = bits(dq_prefix_writes, L, ac, dq_kt)
        assert bits(dq_carry_reads, L, ac, dq_kt) & ~written_carry == 0, f"dQ reads an unwritten product, L={L}"
        carry, prefix = bits(dkv_reads, L, ac, dkv)
        assert carry & ~written_carry == 0, f"dK/dV reads an unwritten product, L={L}"
        assert prefix & ~written_prefix == 0, f"dK/dV reads an unwritten prefix sum, L={L}"


@pytest.mark.parametrize("L,dq_kt,dkv", [(33, 32, "pipelined128"), (161, 32, "pipelined128"), (97, 32, "producer64"),
                                          (97, 32, "wave")])
def test_model_flags_a_skip_test_that_counts_rows_beyond_the_end(L, dq_kt, dkv):
    """A skip test that lets rows beyond the sequence's end count as seeing a sub-tile (`jb > w_last - 1`) reads
    prefix sums the dQ kernel never wrote when L - 1 is a multiple of 32 but not of 128: the model must tell the two
    skip tests apart, or it pins nothing."""
    written_prefix = dq_prefix_writes(L, 0, dq_kt)
    assert not dkv_reads(L, 0, dkv, rows_beyond_end_count=True)[1] <= written_prefix
    assert dkv_reads(L, 0, dkv)[1] <= written_prefix


def test_key_tiles_ask_for_no_row_outside_their_sequence():
    """Key tiles (csrc/sba_bwd_chain.hip) fetch a row block's scalars ahead: blocks 0 and 1 of the next tile while the one before ends, block
    s + 2 in slot s.  Block k is rows 32 (nb - 1 - k) on; a tile of one block has no block 1 (its rows would lie in front of the sequence)."""
    for L in range(1, 700):
        nb = cdiv(L, 32)
        for J in range(cdiv(L, 128)):
            n = nb - 4 * J
            fetched = [k for k in (0, 1) if n > k] + [s + 2 for s in range(n) if s + 2 < n]
            assert sorted(fetched) == list(range(n))
            assert all(128 * J <= 32 * (nb - 1 - k) < L for k in fetched), (L, J)
