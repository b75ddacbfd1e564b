"""Which backward a call runs, and in which groups of heads, under workspace limits: a group on row tiles has to fill the chip and its
eight XCDs by itself, as a call of its own would."""
import ctypes

import pytest

from stickbreaking_attention import _native

pytestmark = pytest.mark.gpu

TWO_KERNELS, KEY_TILES, ROW_TILES = _native.TWO_KERNELS, _native.KEY_TILES, _native.ROW_TILES


def args(heads, dim, lengths, kernels=0, exact=False):
    a = _native.SbaArgs()
    a.dtype, a.head_dim, a.num_heads, a.num_seqs = _native.SBA_BF16, dim, heads, len(lengths)
    a.total_tokens, a.max_seqlen, a.backward_kernels = sum(lengths), max(lengths), kernels
    a.row_blocks = sum(8 * -(-n // 256) for n in lengths if n > 256) if exact else 0
    a.cu_seqlens = 256      # (not read: packed sequences; the tensors count as aligned)
    return a


def route(a, workspace):
    a.workspace_bytes = workspace
    return _native.ext().backward_route(ctypes.addressof(a))


def runs_on_row_tiles(heads, dim, lengths, fixed=False, lengths_known=False, add_remainder=False):
    """Whether a call's backward does, for tests that mean to reach it (16-bit data, aligned rows)."""
    a = args(heads, dim, lengths, exact=lengths_known)
    a.add_remainder = int(add_remainder)
    if fixed:
        a.cu_seqlens, a.total_tokens, a.row_blocks = None, lengths[0], 0
    return route(a, 1 << 40) == (ROW_TILES, heads)


LONG, RAGGED, EQUAL = [65536], [16384] + [31] * 600, [4096] * 16


# MB per head on row tiles / the two kernels: LONG 75.6 / 270, RAGGED 40.3 (16.8 with its lengths known) / 38, EQUAL 75.6 at head_dim 128, 37.8 at 64
@pytest.mark.parametrize("heads,dim,lengths,megabytes,exact,expected", [
    (8, 128, LONG, 620, False, (ROW_TILES, 8)),       # (less than the whole call asks for, which the two kernels could run in as well)
    (8, 128, LONG, 330, False, (TWO_KERNELS, 1)),     # 4 + 4 heads of one sequence: four queues, four XCDs
    (32, 128, LONG, 1600, False, (ROW_TILES, 16)),    # 16 + 16
    (40, 128, LONG, 2990, False, (ROW_TILES, 32)),    # 32 + 8, not 20 + 20
    (15, 128, LONG, 1100, False, (ROW_TILES, 8)),     # 8 + 7
    (32, 128, RAGGED, 370, False, (ROW_TILES, 32)),   # (launches of 8 heads share the memory)
    (32, 128, RAGGED, 210, False, (TWO_KERNELS, 5)),  # the long sequence is most of the work
    (32, 128, RAGGED, 150, True, (ROW_TILES, 32)),
    (12, 128, EQUAL, 320, False, (ROW_TILES, 4)),     # many sequences: the queues even out over them
    (12, 64, EQUAL, 195, False, (ROW_TILES, 4)),
    (16, 128, [512] * 32, 50, False, (TWO_KERNELS, 16)),      # 2 heads: tiles for half the compute units
])
def test_groups_of_heads(gpu_device, heads, dim, lengths, megabytes, exact, expected):
    a = args(heads, dim, lengths, exact=exact)
    assert route(a, 1 << 40) == (ROW_TILES, heads)
    assert route(a, megabytes * 1000 * 1000) == expected


def test_other_forms(gpu_device):
    for a, expected in ((args(32, 128, [1024] * 32, kernels=1), (TWO_KERNELS, 32)), (args(8, 128, [2048, 2048]), (KEY_TILES, 8)),
                        (args(12, 64, [200] * 8), (TWO_KERNELS, 12)), (args(12, 128, [12288]), (ROW_TILES, 8))):      # (8 + 4)
        assert route(a, 1 << 40) == expected


@pytest.mark.parametrize("a,form,count", [
    (args(12, 64, [64, 3, 50]), _native.TINY, 1), (args(8, 128, [64] * 4), _native.TINY, 1), (args(12, 50, [64, 3], kernels=1), _native.TINY, 1),
    (args(8, 128, [64] * 4, kernels=2), KEY_TILES, 1),                                    # (which takes no tiny ones apart)
    (args(12, 7, [64, 3]), TWO_KERNELS, 2), (args(12, 64, [65, 3]), TWO_KERNELS, 2),
    (args(32, 64, [20] * 300 + [70]), TWO_KERNELS, 3),
    (args(16, 128, [8] * 70 + [200]), KEY_TILES, 2),                                      # apart from key tiles, under 12 K rows x heads
    (args(32, 128, [20] * 300 + [4000]), ROW_TILES, 3),                                   # (the clearing kernel is one)
    (args(32, 128, [20] * 300 + [4000], kernels=1), TWO_KERNELS, 3)])
def test_tiny_sequences_are_reported(gpu_device, a, form, count):
    assert route(a, 1 << 40) == (form, a.num_heads)
    assert _native.lib().sba_bwd_kernels(ctypes.byref(a)) == count
