"""A CPU model of the one-wave-per-SIMD loop (csrc/det_gemm_solo.h): where its loads go in memory and in LDS, the rows its lanes
read back, and the order in which the five parts of the LDS are filled and read."""

from __future__ import annotations

import pytest

U32 = 1 << 32
LOADS, PART = 8, 256 * 128


def plain_row(r, last, _half):
    return min((r & ~63) + ((r & 15) >> 2) * 16 + ((r >> 4) & 3) * 4 + (r & 3), last)


def gated_row(r, last, half):
    return min((r >> 7) * 64 + ((r & 15) >> 2) * 16 + ((r >> 4) & 3) * 4 + (r & 3), last) + ((r >> 6) & 1) * half


def token_row(r, last, _half):
    return min(r, last)


def loads(row_of, last, half, ld):
    """(LDS byte offset in the part, byte offset from the tile's first row, row) of every lane of every load of a part."""
    for wave in range(4):
        for j in range(LOADS):
            for lane in range(64):
                row = row_of(wave * 64 + j * 8 + (lane >> 3), last, half)
                off = (row * ld * 2 + ((lane & 7) ^ (lane >> 3)) * 16 + (4 - j % 4) * 1024) % U32  # the kernel's 32-bit offset
                at = off + (j % 4) * 1024 - 4 * 1024  # + the instruction's offset, - what the base is moved by
                yield (wave * LOADS + j // 4 * 4 + j % 4) * 1024 + lane * 16, at, row


@pytest.mark.parametrize("row_of,rows,half", [(plain_row, 256, 0), (plain_row, 77, 0), (token_row, 256, 0), (token_row, 1, 0),
                                               (gated_row, 128, 12288), (gated_row, 60, 60)])  # fmt: skip
@pytest.mark.parametrize("ld", [64, 4096, (1 << 23) - 136])
def test_every_lane_reads_inside_its_operand_and_every_chunk_arrives_once(row_of, rows, half, ld):
    if (256 + half) * ld * 2 + 8192 >= U32:
        pytest.skip("solo_offsets_fit() refuses it")
    seen = {}
    for lds, at, row in loads(row_of, rows - 1, half, ld):
        assert 0 <= row < half + rows
        chunk, rest = divmod(at - row * ld * 2, 16)
        assert rest == 0 and 0 <= chunk < 8
        assert lds not in seen and 0 <= lds < PART
        seen[lds] = (row, chunk)
    assert len(seen) == PART // 16
    # what the fragment reads expect: row r, chunk c at r * 128 + 16 (c ^ (r & 7))
    for r in range(256):
        for c in range(8):
            assert seen[r * 128 + 16 * (c ^ (r & 7))] == (row_of(r, rows - 1, half), c)


@pytest.mark.parametrize("spans", ["plain", "gated"])
def test_a_lane_owns_sixteen_consecutive_features(spans):
    row_of = plain_row if spans == "plain" else gated_row
    for wave_n in range(2):
        for grp in range(4):
            for h in range(2):
                # MFMA tile 4 h + jn of the wave, accumulator row 4 grp + q
                run = [row_of(wave_n * 128 + (4 * h + jn) * 16 + 4 * grp + q, 10**6, 10**7) for jn in range(4) for q in range(4)]
                first = wave_n * 128 + h * 64 + grp * 16 if spans == "plain" else wave_n * 64 + grp * 16 + h * 10**7
                assert run == list(range(first, first + 16))


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


def kmajor_swizzle(k_row):
    return 4 * ((k_row >> 1) & 1) + 2 * (((k_row >> 3) ^ (k_row >> 4)) & 1)


def kmajor_loads(rows, k_left, ld):
    """The same of a K-major operand: rows its matrix has from the tile's first one on, K values left from the K tile's first one on."""
    for wave in range(4):
        for j in range(LOADS):
            for lane in range(64):
                rib = lane >> 3
                first = wave * 64 + ((lane & 7) ^ (4 * ((rib >> 1) & 1))) * 8
                off = (rib * ld * 2 + min(first ^ (((j ^ (j >> 1)) & 1) * 16), rows - 8) * 2) % U32
                scalar = ld * 16 * j + 4 * 1024 - (j % 4) * 1024
                lds = (wave * LOADS + j) * 1024 + lane * 16
                outside = rib >= k_left - 8 * j
                yield lds, (0x80000000 if outside else off), scalar, (j % 4) * 1024


@pytest.mark.parametrize("rows", [256, 264, 200, 8])
@pytest.mark.parametrize("k_left", [64, 24, 1, 63])
@pytest.mark.parametrize("ld", [264, 4096, 151936, (1 << 23) - 8])
def test_kmajor_columns_arrive_once_and_are_read_where_they_lie(rows, k_left, ld):
    span = 0x7FFF0000  # what the hardware takes as inside the buffer, which begins 4 KiB before the operand
    seen = {}
    for lds, off, scalar, imm in kmajor_loads(rows, k_left, ld):
        assert lds not in seen and 0 <= lds < PART
        if off >= span - scalar - imm:
            assert off == 0x80000000
            seen[lds] = None  # zeros
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
