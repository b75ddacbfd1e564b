"""CPU checks of the backward on row tiles (csrc/sba_bwd_row.hip): which recorded products it reads, how the queues of its tiles fall, and
what its inline assembly has to keep that the compiler does not check."""
import ctypes
import heapq
import os
import random
import re
import shutil
import subprocess

import pytest

from test_carry_slots_model import bits, cdiv, forward_writes, slot

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "stickbreaking-attention_amd", "csrc")


def row_tile_reads(L, ac):
    """Products used by the 32 rows of a wave against a 32-key block: slots (block, row), rows beyond the sequence as its last one."""
    m, out = cdiv(L, 128), set()
    for q0 in range(0, L, 256):
        for w_first in range(q0, min(q0 + 256, L), 32):
            last_seen = min(w_first + 31, L - 1) - 1 + ac
            for u in range(last_seen // 32 + 1 if last_seen >= 0 else 0):
                for row in range(w_first, w_first + 32):
                    out.add(slot(u, min(row, L - 1), m))
    return out


@pytest.mark.parametrize("fwd_kt", [32, 64, "split"])
@pytest.mark.parametrize("ac", [0, 1])
def test_every_product_read_was_written(fwd_kt, ac):
    for L in list(range(1, 300)) + [511, 512, 513, 640, 641, 673, 705, 1000]:
        assert bits(row_tile_reads, L, ac) & ~bits(forward_writes, L, ac, fwd_kt) == 0, f"L={L}"


def test_tiles_are_laid_from_the_end():
    """Row tiles of a sequence: every row, and every block of 32 keys, is in one; the keys a tile sweeps are those it, or the tiles below it,
    own, and those it hands down belong to the tiles below; the tile above sweeps 8 blocks more."""
    for L in range(1, 1400):
        rows, blocks, above = [], [], None
        for nth in range(cdiv(L, 256)):
            q_end = cdiv(L, 32) * 32 - 256 * nth
            q0 = max(q_end - 256, 0)
            n, own, waves = q_end // 32, q0 // 32, (q_end - q0) // 32
            assert q_end > q0 and 1 <= waves <= 8 and n == own + waves and (waves == 8 or own == 0)
            assert above is None or above[0] == n + 8 and above[1] == n      # what the tile above hands down are this tile's blocks
            above = n, own
            rows += [r for w in range(waves) for r in range(q0 + 32 * w, min(q0 + 32 * w + 32, L))]
            blocks += range(own, n)
            assert all(q0 + 32 * w < L for w in range(waves))
        assert above[1] == 0 and sorted(rows) == list(range(L)) and sorted(blocks) == list(range(cdiv(L, 32)))


def test_partial_results_of_neighbours_do_not_overlap():
    """The blocks of a sequence start at floor(9 start / 256) of the head's; sequences of up to 256 rows hand nothing over."""
    for L in range(257, 1300):
        for start in range(0, 300):
            first = start * 9 // 256
            assert (start + L) * 9 // 256 - first >= cdiv(L, 32), (L, start)      # before the next sequence's, which starts at or behind
            assert first + cdiv(L, 32) <= (start + L) * 9 // 256 + 2              # within the head's


def test_places_by_slot_do_not_overlap():
    """The list holds sequences with more query tiles of 128 rows first; one of more than 256 rows has 8 key blocks per row tile at 8 times
    its first slot, all within SbaArgs.row_blocks."""
    rng = random.Random(0)
    for _ in range(300):
        lengths = [rng.choice([0, 1, 255, 256, 257, 511, 512, 513, rng.randint(1, 3000)]) for _ in range(rng.randint(1, 40))]
        total, slot0, end = sum(8 * cdiv(n, 256) for n in lengths if n > 256), 0, 0
        for n in sorted(lengths, key=lambda n: -cdiv(n, 128)):
            if n > 256:
                assert 8 * slot0 >= end      # behind the one before
                end = 8 * slot0 + cdiv(n, 256) * 8 - 8      # (its last tile's own rows are handed to none)
                assert end <= total
            slot0 += cdiv(n, 256)


@pytest.mark.parametrize("turns", [1, 2, 3, 5, 8])
def test_tiles_that_take_turns(turns):
    """Places in the list (forward_service in csrc/sba_sched.hpp): each is taken once, the tile above comes first, and in a group those with
    most keys do."""
    rng = random.Random(turns)
    for _ in range(200):
        lengths = [rng.choice([0, 1, 256, 257, 512, 513, rng.randint(1, 5000)]) for _ in range(rng.randint(1, 64))]
        order = sorted(range(len(lengths)), key=lambda s: -cdiv(lengths[s], 128))
        nk = [cdiv(lengths[s], 256) for s in order if lengths[s]]      # by rank
        first = [sum(nk[:r]) for r in range(len(nk))]
        at = {}
        for rank, n in enumerate(nk):
            group = rank // turns * turns
            members = [nk[r] if r < min(group + turns, len(nk)) else 0 for r in range(group, group + 8)]
            for t in range(n):
                place = first[group] + (rank - group) + sum(max(0, m - (n - t)) for m in members)
                assert place not in at
                at[place] = (rank, t, n - t, group)
        assert sorted(at) == list(range(sum(nk)))
        where = {v[:2]: k for k, v in at.items()}
        for (rank, t), k in where.items():
            assert t == 0 or where[rank, t - 1] < k
        for k in range(1, len(at)):
            assert at[k][3] >= at[k - 1][3] and (at[k][3] > at[k - 1][3] or at[k][2] <= at[k - 1][2])
    for seqs, n in ((1, 3), (4, 32), (9, 1), (17, 5)):      # equal lengths
        places = sorted(s // turns * turns * n + t * min(turns, seqs - s // turns * turns) + s % turns for s in range(seqs) for t in range(n))
        assert places == list(range(seqs * n))


@pytest.mark.parametrize("heads", [1, 4, 7, 8, 12, 20, 32])
def test_every_head_is_in_one_queue(heads):
    """... of every sequence, and 8 sequences in a row fill the queues alike."""
    per_slot, units = cdiv(heads, 8), [0] * 8
    for rank in range(16):
        first = (rank ^ rank >> 1) * heads      # (Gray code)
        by_queue = [[h for i in range(per_slot) for h in [((q - first) % 8) + 8 * i] if h < heads] for q in range(8)]
        assert sorted(sum(by_queue, [])) == list(range(heads))
        units = [u + len(b) for u, b in zip(units, by_queue)]
        if rank % 8 == 7:
            assert max(units) - min(units) <= heads % 8, (rank, units)


def test_tiles_of_a_queue_stay_on_one_xcd():
    """Whatever XCDs the workgroups of a queue land on: those that are not where the first one is leave, the others take every tile, in list
    order, so that a tile never waits for one that nobody has taken."""
    rng = random.Random(0)
    for _ in range(200):
        workgroups = [rng.randint(1, 8) if rng.random() < 0.5 else 1 for _ in range(rng.randint(1, 32))]      # XCD + 1, in order of arrival
        recorded, stay = 0, []
        for xcd in workgroups:      # compare and swap
            recorded = recorded or xcd
            if xcd == recorded:
                stay.append(xcd)
        assert stay and set(stay) == {recorded}
        cursor, taken = 0, []
        busy = [0] * len(stay)
        while cursor < 100:      # whoever is free takes the next one; tile t waits for t - 1, which was taken before it
            w = min(range(len(stay)), key=lambda i: busy[i])
            taken.append(cursor)
            busy[w] += rng.randint(1, 9)
            cursor += 1
        assert taken == list(range(100))


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    """The functions of csrc/sba_params.hpp that say how much work a sequence is and how many workgroups begin with sequences of one tile."""
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no g++")
    folder = tmp_path_factory.mktemp("rules")
    (folder / "rules.cpp").write_text("""#include "sba_params.hpp"
extern "C" uint64_t work(int64_t len) { return sba::row_work(len); }
extern "C" int apart(int wgs, uint64_t single, uint64_t chained, uint64_t longest) {
  return sba::apart_workgroups(wgs, sba::apart_share(single, chained, longest));
}
""")
    subprocess.run([cxx, "-std=c++17", "-O1", "-shared", "-fPIC", "-D__host__=", "-D__device__=", "-I", CSRC, str(folder / "rules.cpp"), "-o",
                    str(folder / "rules.so")], check=True, capture_output=True)
    lib = ctypes.CDLL(str(folder / "rules.so"))
    lib.work.restype, lib.work.argtypes = ctypes.c_uint64, [ctypes.c_int64]
    lib.apart.argtypes = [ctypes.c_int] + 3 * [ctypes.c_uint64]
    return lib


def test_work_of_a_sequence(rules):
    for length in range(0, 3000):
        assert rules.work(length) == sum(cdiv(length, 32) - 8 * nth + 1 for nth in range(cdiv(length, 256))), length


def time_of(wgs, chains, singles, begin_apart):
    """A queue's time until its last tile is done: `begin_apart` workgroups begin with `singles`, all go over to the other list."""
    lists = [list(chains) + (list(singles) if not begin_apart else []), [] if not begin_apart else list(singles)]
    at, free = [0, 0], [(0., i, i >= wgs - begin_apart) for i in range(wgs)]
    heapq.heapify(free)
    end = 0.
    while free:
        now, i, which = heapq.heappop(free)
        end = max(end, now)
        which = which if at[which] < len(lists[which]) else not which
        if at[which] < len(lists[which]):
            heapq.heappush(free, (now + lists[which][at[which]], i, which))
            at[which] += 1
    return end


@pytest.mark.parametrize("chain_cost", [0.9, 1.0, 1.1])
@pytest.mark.parametrize("wgs", [8, 32])
def test_sequences_of_one_tile_do_not_hold_up_the_chains(rules, wgs, chain_cost):
    """The time of a queue with two lists is that of one list, longest first, or up to a seventh more (the tiles of one chain over 20-odd
    workgroups; what runs better side by side, and at the clock that idle workgroups leave, is not in here), whatever there is beside many short
    sequences, and also if the tiles of chains take 10 % more or less than the rule believes."""
    rng = random.Random(wgs)
    batches = [([1024], 2048, 64), ([2048], 2048, 64), ([600], 1000, 64), ([1500] * 3, 300, 100), ([16384], 2048, 32), ([16384], 2048, 64),
               ([12000], 150, 250), ([700] * 8, 500, 60), ([5000] * 4, 1000, 40), ([8192], 300, 64), ([4096, 3000], 200, 100)]
    batches += [([rng.randint(257, rng.choice([1000, 16384])) for _ in range(rng.choice([1, 1, 2, 5]))], rng.randint(1, 2500), rng.randint(1, 256)) for _ in range(400)]
    two = 0
    for long, n, short in batches:
        single, chained = n * rules.work(short), sum(rules.work(x) for x in long)
        begin_apart = rules.apart(wgs, single, chained, max(rules.work(x) for x in long))
        assert 0 <= begin_apart <= wgs // 2
        two += begin_apart > 0
        chains = [chain_cost * (cdiv(x, 32) - 8 * nth + 1) for x in sorted(long, reverse=True) for nth in range(cdiv(x, 256))]
        singles = [cdiv(short, 32) + 1] * n
        one = time_of(wgs, chains, singles, 0)
        assert time_of(wgs, chains, singles, begin_apart) <= 8 / 7 * one, (long, n, short, begin_apart)
    assert two >= 10      # (and the rule does choose two lists)


@pytest.mark.parametrize("wgs", [1, 2, 5, 32])
def test_two_lists_of_a_queue(wgs):
    """Each workgroup begins with one list and goes over to the other: every claim below `all` is handed out once, those of the chains in order."""
    rng = random.Random(wgs)
    for _ in range(200):
        chained, single = rng.choice([0, 1, 7, 40]), rng.choice([0, 1, 9, 300])
        both, begin_apart = chained + single, (wgs * rng.randrange(0, 1025) + 512) >> 10
        if not begin_apart:
            chained = both      # one list holds all
        cursor, out = [0, 0], []
        apart = [i >= wgs - begin_apart and chained < both for i in range(wgs)]
        running = set(range(wgs))
        while running:
            i = rng.choice(sorted(running))
            first = apart[i]
            c = cursor[first] + (chained if first else 0)
            cursor[first] += 1
            if c >= (both if first else chained):
                c = both
                if chained > 0 if first else chained < both:
                    c = cursor[not first] + (0 if first else chained)
                    cursor[not first] += 1
                    if c >= (chained if first else both):
                        c = both
            apart[i] = c >= chained
            if c >= both:
                running.discard(i)
            else:
                out.append(c)
        assert sorted(out) == list(range(both))
        assert [c for c in out if c < chained] == list(range(chained))


@pytest.fixture(scope="module")
def listing(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    flags = re.search(r"^HIPFLAGS = (.*?)\nSRCS", open(os.path.join(CSRC, "Makefile")).read(), re.S | re.M).group(1)
    flags = flags.replace("\\\n", " ").replace("$(ARCH)", "gfx950").split()
    out = str(tmp_path_factory.mktemp("s") / "row.s")
    subprocess.run([hipcc, *flags, "-S", "--cuda-device-only", os.path.join(CSRC, "sba_bwd_row.hip"), "-o", out], check=True, capture_output=True)
    kernels, name = {}, None
    for line in open(out):
        m = re.match(r"(_Z\w+):", line)
        if m:
            name = m.group(1)
            kernels[name] = []
        if name:
            kernels[name].append(line)
        if ".Lfunc_end" in line:
            name = None
    return {n: k for n, k in kernels.items() if "bwd_row_kernel" in n}


def registers(text, kind):
    out = set()
    for a, b, c in re.findall(rf"\b{kind}(\d+)\b|\b{kind}\[(\d+):(\d+)\]", text):
        out |= {int(a)} if a else set(range(int(b), int(c) + 1))
    return out


VECTOR_MEMORY = re.compile(r"global_|buffer_(load|store)|scratch_|flat_")


def test_scalars_of_vector_memory_instructions_are_old_enough(listing):
    """A scalar register written by a vector instruction (a reloaded spill) may be read by a vector-memory instruction only five wait
    states later, which the compiler keeps for its own instructions and not for those in inline assembly."""
    assert listing
    for name, lines in listing.items():
        age = {}
        for line in lines:
            text = line.split(";")[0].strip()
            if not text or text.endswith(":") or text.startswith("."):
                continue
            op, _, rest = text.partition(" ")
            if VECTOR_MEMORY.match(op):
                young = [r for r in registers(text, "s") if age.get(r, 9) < 5]
                assert not young, f"{name}: {text}: s{young}"
            step = int(rest, 0) + 1 if op == "s_nop" else 1
            age = {r: a + step for r, a in age.items() if a + step < 6}
            written = registers(rest.split(",")[0], "s")
            if op in ("v_readlane_b32", "v_readfirstlane_b32") or op.startswith("v_cmp"):
                age.update((r, 0) for r in written)
            elif op.startswith("s_") and not op.startswith(("s_waitcnt", "s_cmp", "s_cbranch", "s_barrier", "s_nop", "s_branch")):
                for r in written:
                    age.pop(r, None)


def test_registers_on_their_way_are_left_alone(listing):
    """No register that a load in inline assembly is still filling is read, copied or spilled before a wait that covers the load.
    Forward over the control-flow graph: register -> fewest vector-memory operations issued since its load, over all paths; "nothing
    in flight" marks the head of the loop, where by construction nothing is."""
    for name, lines in listing.items():
        order, blocks, asm = ["entry"], {"entry": []}, False
        for line in lines:
            if "#ASMSTART" in line or "#ASMEND" in line:
                asm = "#ASMSTART" in line
                continue
            m = re.match(r"(\.LBB\d+_\d+):", line)
            if m:
                order.append(m.group(1))
                blocks[m.group(1)] = []
                continue
            text = "nothing in flight" if "nothing in flight" in line else line.split(";")[0].strip()
            if text and not text.startswith(".") and not text.endswith(":"):
                blocks[order[-1]].append((text, asm))
        follow = dict(zip(order, order[1:]))
        state, work, bad = {"entry": {}}, ["entry"], []

        def flow(to, s):
            old = state.get(to)
            new = dict(s) if old is None else {r: min(old.get(r, 99), s.get(r, 99)) for r in {**old, **s}}
            if new != old:
                state[to] = new
                work.append(to)

        def run(block, visit):
            s = dict(state[block])
            for text, in_asm in blocks[block]:
                op, _, rest = text.partition(" ")
                if text == "nothing in flight":
                    s = {}
                elif op.startswith(("s_cbranch", "s_branch")):
                    visit(rest.strip(), s)
                    if op == "s_branch":
                        return
                elif op == "s_endpgm":
                    return
                elif op == "s_waitcnt":
                    m = re.search(r"vmcnt\((\d+)\)", rest)
                    s = {r: c for r, c in s.items() if c < int(m.group(1))} if m else s
                else:
                    if not op.startswith("s_") and registers(text, "v") & set(s):
                        bad.append(f"{block}: {text}")
                    if VECTOR_MEMORY.match(op):
                        s = {r: min(c + 1, 63) for r, c in s.items()}
                        if in_asm and "_load_" in op and " lds" not in text:
                            s.update((r, 0) for r in registers(rest.split(",")[0], "v"))
            if block in follow:
                visit(follow[block], s)

        while work:
            run(work.pop(), flow)
        bad.clear()
        for block in state:
            run(block, lambda *_: None)
        assert not bad, f"{name}: {bad[:5]}"


def test_stored_registers_outlive_their_store_by_a_wait_state(listing):
    """The hardware reads the data of a store of more than 8 bytes a wait state after it was issued: a vector instruction that writes those
    registers must not be the next one.  The compiler keeps this for its own stores and not for those in inline assembly."""
    for name, lines in listing.items():
        data = set()
        for line in lines:
            text = line.split(";")[0].strip()
            if not text or text.endswith(":") or text.startswith("."):
                continue
            op, _, rest = text.partition(" ")
            if op.startswith("v_") and not op.startswith(("v_cmp", "v_readlane", "v_readfirstlane")):
                assert not registers(re.split(r",(?![^\[]*\])", rest)[0], "v") & data, f"{name}: {text}"
            wide = re.match(r"(global|buffer|scratch)_store_dwordx[34]", op)
            data = registers(re.split(r",(?![^\[]*\])", rest)[1 if op.startswith(("global", "scratch")) else 0], "v") if wide else set()
