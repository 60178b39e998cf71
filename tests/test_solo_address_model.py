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
