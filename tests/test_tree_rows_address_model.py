"""A CPU model of the lane addresses of det_gemm_tree_rows_kernel (csrc/det_gemm_tree.hip), both row counts and leaf
lengths: every global address lies inside its operand, every granule of a leaf is loaded once, every lane reads from LDS
the row, column and k that it is to hold, and all of it stays inside the wave's region."""

from __future__ import annotations

import itertools

import pytest


def swizzle(pair: int, chunks: int) -> int:
    return (pair >> 2) & 3 if chunks == 4 else 0


@pytest.mark.parametrize("r", [1, 2])
@pytest.mark.parametrize("m, n, k, depth", [(1, 64, 1024, 5), (16, 100, 768, 5), (33, 257, 4096, 7), (200, 130, 12288, 9),
                                            (47, 70, 32768, 10), (32, 128, 3072, 7)])  # fmt: skip
@pytest.mark.parametrize("extra", [0, 40])
def test_every_lane_address_lies_inside_its_operand(r, m, n, k, depth, extra):
    split, leaf = (3 if r == 1 else 2), k >> depth
    chunks, rows, waves = leaf // 8, 16 * r, 1 << split
    leaves = 1 << (depth - split)
    assert leaves >= 4 and leaves % 4 == 0 and waves * leaves * leaf == k
    sets = 4 // r
    a_pitch, b_pitch = k + extra, k + 2 * extra
    a_elems, b_elems = (m - 1) * a_pitch + k, (n - 1) * b_pitch + k
    a_bytes, leaf_bytes = 1024 * r, 1024 * (r + chunks)
    row_groups = -(-m // rows)
    groups = -(-n // 64) * row_groups
    for gid, wave, which in itertools.product({0, row_groups - 1, groups - 1}, {0, waves - 1}, {0, leaves - 1}):
        n0, m0 = (gid // row_groups) * 64, (gid % row_groups) * rows
        at = wave * leaves * leaf + which * leaf
        lds = {}  # byte offset in the leaf's region -> (operand, row or column, first k)
        for j, lane in itertools.product(range(chunks), range(64)):
            g = 64 * j + lane
            col, chunk = g // chunks, (g % chunks) ^ swizzle(g // chunks, chunks)
            col_in = col if n0 + col < n else n - 1 - n0
            first = n0 * b_pitch + at + col_in * b_pitch + 8 * chunk
            assert 0 <= first and first + 8 <= b_elems
            lds[a_bytes + 1024 * j + 16 * lane] = ("w", col, 8 * chunk)
        for j, lane in itertools.product(range(r), range(64)):
            g = min(64 * j + lane, rows * chunks - 1)
            row, chunk = g // chunks, (g % chunks) ^ swizzle(g // chunks, chunks)
            row_in = row if m0 + row < m else m - 1 - m0
            first = m0 * a_pitch + at + row_in * a_pitch + 8 * chunk
            assert 0 <= first and first + 8 <= a_elems
            place = 1024 * j + 16 * lane
            assert place + 16 <= a_bytes
            lds[place] = ("a", row, 8 * chunk)
        for lane in range(64):
            for c in range(chunks):
                assert lds[a_bytes + lane * 16 * chunks + 16 * (c ^ swizzle(lane, chunks))] == ("w", lane, 8 * c)
            for i in range(-(-chunks // sets)):
                row, chunk = lane % rows, min(sets * i + lane // rows, chunks - 1)
                assert lds[row * 16 * chunks + 16 * (chunk ^ swizzle(row, chunks))] == ("a", row, 8 * chunk)
        # block set * r + g of the instruction's row operand (lanes 16 b .. 16 b + 15) holds row group g at chunk sets i + set
        for i, s, g in itertools.product(range(-(-chunks // sets)), range(sets), range(r)):
            if sets * i + s < chunks:
                lanes = range(16 * (s * r + g), 16 * (s * r + g) + 16)
                assert [(x % rows, min(sets * i + x // rows, chunks - 1)) for x in lanes] == [
                    (16 * g + q, sets * i + s) for q in range(16)]  # fmt: skip
        assert max(lds) + 16 <= leaf_bytes
    assert 2 * waves * leaf_bytes * 2 <= 160 * 1024  # two workgroups per CU
    assert 2 * waves * leaf_bytes >= waves * 8 * r * 64 * 4  # the fold's table
