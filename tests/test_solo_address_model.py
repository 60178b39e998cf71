"""A CPU model of the one-wave-per-SIMD loop (csrc/det_gemm_solo.h): where its loads go in memory and in LDS, the rows its lanes
read back, and the order in which the five parts of the LDS, or the stages of a ring, are filled and read."""

from __future__ import annotations

import pytest

U32 = 1 << 32
LOADS, PART = 8, 256 * 128


def plain_row(tn):
    """SoloPlainRows: 16 tn rows a wave, spans of 64 whose lane groups have 16 consecutive features; of 96 the last 32 are half a span."""

    def feature(r):
        in_wave = r % (16 * tn)
        span = in_wave & ~63
        run = 8 if (16 * tn) % 64 and span + 64 > 16 * tn else 16
        return r - in_wave + span + ((r & 15) >> 2) * run + (((in_wave - span) >> 4) & 3) * 4 + (r & 3)

    return lambda r, last, _half: min(feature(r), last)


def gated_row(tn, split=False):
    """SoloGatedRows: half of a wave's rows gate, half up rows of the same features."""

    def row(r, last, half):
        wave, tile = r // (16 * tn), r % (16 * tn) // 16
        f = wave * 8 * tn + ((r & 15) >> 2) * (2 * tn) + tile % (tn // 2) * 4 + (r & 3)
        return min(f, last) + (0 if split else tile // (tn // 2) * half)

    return row


def token_row(r, last, _half):
    return min(r, last)


def loads(row_of, part_rows, last, half, ld):
    """(LDS byte offset in the part, byte offset from the tile's first row, row) of every lane of every load of a part."""
    count = part_rows // 32  # of a wave
    for wave in range(4):
        for j in range(count):
            for lane in range(64):
                row = row_of(wave * 8 * count + j * 8 + (lane >> 3), last, half)
                off = (row * ld * 2 + ((lane & 7) ^ (lane >> 3)) * 16 + (4 - j % 4) * 1024) % U32  # the kernel's 32-bit offset
                at = off + (j % 4) * 1024 - 4 * 1024  # + the instruction's offset, - what the base is moved by
                yield (wave * count + j // 4 * 4 + j % 4) * 1024 + lane * 16, at, row


# (row map, rows of the part, rows that the matrix has from the tile's first one on, rows between gate and up)
MAPS = [
    (plain_row(8), 256, 256, 0), (plain_row(8), 256, 77, 0), (plain_row(6), 192, 192, 0), (plain_row(6), 192, 100, 0),
    (token_row, 256, 256, 0), (token_row, 192, 1, 0), (token_row, 128, 128, 0), (gated_row(8), 256, 128, 12288), (gated_row(8), 256, 60, 60),
    (gated_row(6), 192, 96, 3072), (gated_row(4), 128, 64, 3072), (gated_row(4), 128, 33, 33), (gated_row(2), 64, 32, 3072),
    (gated_row(8, True), 256, 128, 0), (gated_row(6, True), 192, 50, 0), (gated_row(2, True), 64, 32, 0),
]  # fmt: skip


@pytest.mark.parametrize("row_of,part,rows,half", MAPS)
@pytest.mark.parametrize("ld", [64, 4096, (1 << 23) - 136])
def test_every_lane_reads_inside_its_operand_and_every_chunk_arrives_once(row_of, part, rows, half, ld):
    if (256 + half) * ld * 2 + 8192 >= U32:
        pytest.skip("solo_offsets_fit() refuses it")
    seen = {}
    for lds, at, row in loads(row_of, part, rows - 1, half, ld):
        assert 0 <= row < half + rows
        chunk, rest = divmod(at - row * ld * 2, 16)
        assert rest == 0 and 0 <= chunk < 8
        assert lds not in seen and 0 <= lds < part * 128
        seen[lds] = (row, chunk)
    assert len(seen) == part * 128 // 16
    # what the fragment reads expect: row r, chunk c at r * 128 + 16 (c ^ (r & 7))
    for r in range(part):
        for c in range(8):
            assert seen[r * 128 + 16 * (c ^ (r & 7))] == (row_of(r, rows - 1, half), c)


@pytest.mark.parametrize("spans,tn", [("plain", 8), ("plain", 6), ("gated", 8), ("gated", 6), ("gated", 4), ("gated", 2)])
def test_a_lane_owns_consecutive_features(spans, tn):
    """What the stores take for granted: the MFMA tiles of a run are one lane's consecutive features, and all of a wave's are there."""
    up = 10**7
    row_of = plain_row(tn) if spans == "plain" else gated_row(tn)
    for wave_n in range(2):
        seen = []
        for grp in range(4):
            if spans == "plain":  # (first MFMA tile, tiles, first feature of the wave's)
                runs = [(4 * h, 4, 64 * h + 16 * grp) for h in range(tn // 4)] + ([(tn - 2, 2, tn // 4 * 64 + 8 * grp)] if tn % 4 else [])
                base = wave_n * 16 * tn
            else:
                runs = [(0, tn // 2, grp * 2 * tn), (tn // 2, tn // 2, grp * 2 * tn + up)]
                base = wave_n * 8 * tn
            for first_tile, tiles, first in runs:
                # MFMA tile of the wave, accumulator row 4 grp + q
                run = [row_of(wave_n * 16 * tn + (first_tile + t) * 16 + 4 * grp + q, 10**6, up) for t in range(tiles) for q in range(4)]
                assert run == list(range(base + first, base + first + 4 * tiles))
                seen += run
        assert len(set(seen)) == 16 * tn


@pytest.mark.parametrize("tn", [8, 6, 4, 2])
def test_a_wave_loads_gate_rows_or_up_rows(tn):
    """With two weights a wave's loads have one base: even waves the gate weight's, odd ones the up weight's."""
    for r in range(32 * tn):
        wave = r // (8 * tn)
        assert (gated_row(tn)(r, 10**6, 10**7) >= 10**7) == bool(wave & 1)


@pytest.mark.parametrize("k_tiles,tiles", [(1, 1), (1, 4), (2, 3), (3, 2), (7, 2)])
def test_no_part_is_overwritten_before_it_is_read(k_tiles, tiles):
    """Parts are named (output tile, K tile, operand). A load may land at any moment from its issue to the wait that covers it."""
    stream = [(o, k) for o in range(tiles) for k in range(k_tiles)]
    place = [None] * 5  # what lies there, or is on its way
    landed = set()
    waiting = []  # issued and not waited for, in order
    head = 0

    def issue(operand, slot):
        part = (head, operand)
        place[slot] = part
        waiting.append(part)

    def wait(keep):
        while len(waiting) > keep:
            landed.add(waiting.pop(0))

    for t in range(2):
        issue("w", 2 * t)
        issue("x", 2 * t + 1)
        head += 1
    wait(2)
    w, x, spare = 0, 1, 4
    nxt = lambda s: (s + 1) % 5  # noqa: E731
    for i in range(len(stream)):
        for operand, slot in (("w", w), ("x", x)):  # both K steps of tile i are read before the barrier of its second step
            assert place[slot] == (i, operand) and (i, operand) in landed
        issue("w", spare)  # under the first step: the place of token rows that every wave has read
        for operand, slot in (("w", w), ("x", x)):
            assert place[slot] == (i, operand)
        wait(1)  # all but the youngest part, then the barrier
        old_w = w
        spare, w = x, nxt(x)
        x = nxt(w)
        issue("x", old_w)
        head += 1


@pytest.mark.parametrize("bn,bm", [(192, 192), (256, 128), (192, 128), (128, 192), (128, 128), (64, 192), (64, 128)])
@pytest.mark.parametrize("k_tiles,tiles", [(1, 1), (1, 4), (2, 3), (3, 2), (9, 2)])
def test_no_stage_of_a_ring_is_overwritten_before_it_is_read(bn, bm, k_tiles, tiles):
    """Smaller shapes: a ring of stages of a whole K tile, token rows a step behind weight rows; waits count load instructions."""
    stage_bytes = (bn + bm) * 128
    stages = 5 * PART // stage_bytes
    assert stages >= 3
    of = {"w": bn // 32, "x": bm // 32}  # load instructions of a wave
    ahead = (stages - 2) * (of["w"] + of["x"])
    place = {}
    landed, waiting = set(), []
    head = 0

    def issue(operand, stage):
        place[(stage, operand)] = (head, operand)
        waiting.extend([(head, operand)] * of[operand])

    def wait(keep):
        assert keep <= 63  # the counter's range
        while len(waiting) > keep:
            part = waiting.pop(0)
            if part not in waiting:
                landed.add(part)

    for t in range(stages - 1):
        issue("w", t)
        issue("x", t)
        head += 1
    issue("w", stages - 1)
    wait(ahead + of["w"])
    at, spare = 0, stages - 1
    for i in range(k_tiles * tiles):
        read = [((at, operand), (i, operand)) for operand in ("w", "x")]
        assert all(place[where] == part and part in landed for where, part in read)  # its first step's fragments are in registers
        issue("x", spare)  # under the first step, in which the second one's fragments are read
        head += 1
        assert all(place[where] == part for where, part in read)
        wait(ahead)  # then the barrier: the next K tile has landed, and no wave reads this one any more
        spare, at = at, (at + 1) % stages
        issue("w", spare)


def kmajor_swizzle(k_row):
    return 4 * ((k_row >> 1) & 1) + 2 * (((k_row >> 3) ^ (k_row >> 4)) & 1)


def kmajor_loads(rows, k_left, ld):
    """(LDS byte offset, lane offset, scalar offset, instruction offset) of a K-major operand, and the size of the buffer that begins
    4 KiB before it: rows its matrix has from the tile's first one on, K values left from the K tile's first one on."""
    size = ld * 2 * min(k_left, 64) + 4 * 1024
    for wave in range(4):
        for j in range(LOADS):
            for lane in range(64):
                rib = lane >> 3
                first = wave * 64 + ((lane & 7) ^ (4 * ((rib >> 1) & 1))) * 8
                off = (rib * ld * 2 + min(first ^ (((j ^ (j >> 1)) & 1) * 16), rows - 8) * 2) % U32
                scalar = min((ld * 16 * j + 4 * 1024 - (j % 4) * 1024) % U32, size)
                yield (wave * LOADS + j) * 1024 + lane * 16, off, scalar, (j % 4) * 1024, size


@pytest.mark.parametrize("rows", [256, 264, 200, 8])
@pytest.mark.parametrize("k_left", [64, 24, 1, 63, 1000])
@pytest.mark.parametrize("ld", [264, 4096, 151936, (1 << 23) - 8])
def test_kmajor_columns_arrive_once_and_are_read_where_they_lie(rows, k_left, ld):
    seen = {}
    for lds, off, scalar, imm, size in kmajor_loads(rows, k_left, ld):
        assert lds not in seen and 0 <= lds < PART
        assert 0 <= scalar <= size < U32  # or the check below would wrap
        if off + imm >= size - scalar:  # the hardware's: zeros
            seen[lds] = None
            continue
        k_row, at = divmod(off + scalar + imm - 4 * 1024, ld * 2)
        assert 0 <= k_row < min(64, k_left) and at % 16 == 0 and at // 2 + 8 <= rows
        seen[lds] = (k_row, at // 2)
    assert len(seen) == PART // 16
    # a transposing read: eight bytes of a lane, row tile j16 of a column, K row of its step, lane group and half
    for tile in range(16):
        for k in range(64):
            step, grp, half, a = k // 32, k // 8 % 4, k // 4 % 2, k % 4
            for l4 in range(4):  # the lane's four rows: 4 l4 .. + 3 of the tile
                tr_row = grp * 8 + a
                tr_at = tr_row * 128 + (((l4 >> 1) ^ kmajor_swizzle(tr_row)) << 4) + (l4 & 1) * 8
                place = tile // 4 * 8192 + (tr_at ^ (tile % 4) << 5) + step * 4096 + half * 512
                first = tile * 16 + l4 // 2 * 8
                want = (k, min(first, rows - 8)) if k < k_left else None
                assert seen[place // 16 * 16] == want and place % 16 == (l4 & 1) * 8


@pytest.mark.parametrize("k_rest", [1, 8, 24, 63])
@pytest.mark.parametrize("ld", [264, 4096, (1 << 21) - 8])
def test_chunks_of_a_native_operand_past_the_reduction_read_zeros(k_rest, ld):
    """Beside a K-major operand the last K tile's native chunks behind the reduction get an offset that the buffer does not reach."""
    size, outside = 0x7FFF0000, 0x80000000
    for lds, at, row in loads(token_row, 256, 255, 0, ld):
        j, lane = lds // 1024 % 8, lds % 1024 // 16
        imm = j % 4 * 1024
        off = at - imm + 4 * 1024
        chunk = (lane & 7) ^ (lane >> 3)
        inside = chunk * 8 < k_rest
        assert 0 <= off < outside  # solo_kmajor_fits(): the bit is free
        assert ((off if inside else off | outside) + imm < size) == inside


def shares(na, la, nb, lb, groups):
    """solo_shares(): tiles of the first product and of the second, their lengths in K tiles."""
    rounds, late = divmod(na, groups)
    even = ((na * la + nb * lb) // groups - (rounds + 1) * la) / lb
    best = None
    for t in [0] if even < 0 else [int(even), int(even) + 1]:
        of_late = min(late * t, nb)
        others = -(-(nb - of_late) // (groups - late))
        span = max(rounds * la + others * lb, (rounds + 1) * la + t * lb if late else 0)
        if best is None or span < best[0]:
            best = (span, late, t)
    return best


@pytest.mark.parametrize("na,la,nb,lb", [(128, 70, 256, 38), (272, 2380, 9504, 71), (1, 7, 1, 7), (256, 70, 256, 70), (3, 90, 700, 10), (700, 20, 1, 8)])
def test_two_products_are_shared_out_whole(na, la, nb, lb):
    groups = min(256, na + nb)
    span, late, late_tiles = shares(na, la, nb, lb, groups)
    first, second, longest = [], [], 0
    for g in range(groups):
        of_late = min(late * late_tiles, nb)
        mine = list(range(g, na, groups))
        if g < late:
            more = list(range(g, of_late, late))
        else:
            more = list(range(of_late + g - late, nb, groups - late))
        first += mine
        second += more
        longest = max(longest, len(mine) * la + len(more) * lb)
    assert sorted(first) == list(range(na)) and sorted(second) == list(range(nb)) and longest <= span
    assert span <= (na * la + nb * lb) / groups + la + lb
