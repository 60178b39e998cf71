"""A CPU model of the lane addresses of det_gemm_tree_nodes_kernel (csrc/det_gemm_tree.hip): for launch grids it can be given -
ragged row and column counts, leaves of 24 and of 32, the small ones that the picker gives it and larger ones - every global
address a lane forms lies inside its operand, every 16-byte granule of a wave's leaf of the weight is loaded exactly once for
the columns that exist, and every LDS access stays inside the wave's own staging region. The model restates the
kernel's index arithmetic; it guards that arithmetic's bounds (what a GPU run can only show by faulting), not the
kernel's values, which the GPU tests compare with the oracle. The kernels of 16 and 32 rows per wave have a model of their own."""

from __future__ import annotations

import itertools

import pytest

NODE_SPLIT, NODE_WAVES, MAX_DEPTH, LEAF, COLS, CUS = 3, 8, 10, 32, 16, 256


def tree_depth(k: int) -> int:
    depth, size = 0, k
    while size > LEAF:
        size -= size // 2
        depth += 1
    return depth


def choice(m: int, n: int, k: int) -> str | None:
    """Which node-per-wave kernel det_gemm_tree_launch takes for K-contiguous rows: "nodes", "rows16", "rows32" or none."""
    depth = tree_depth(k)
    if k % (8 << depth) or not 3 < depth <= MAX_DEPTH or (k >> depth) not in (24, 32):
        return None
    groups16, groups32 = -(-n // 64) * -(-m // 16), -(-n // 64) * -(-m // 32)
    turns16, turns32 = -(-groups16 // CUS), -(-groups32 // CUS)
    if 2 * groups16 <= CUS and depth > NODE_SPLIT + 2:
        return "nodes"
    return "rows32" if depth == 4 or (turns32 >= 2 and 48 * turns32 < 25 * turns16) else "rows16"


def swizzle(pair: int, chunks: int) -> int:
    return (pair >> 2) & 3 if chunks == 4 else 0


def model(m: int, n: int, k: int, a_pitch: int, b_pitch: int) -> None:
    depth = tree_depth(k)
    leaf = k >> depth
    chunks = leaf // 8
    row_groups = -(-m // 16)
    leaves = 1 << (depth - NODE_SPLIT - 2)  # under the node of one of the instruction's four blocks
    assert leaves >= 2 and leaves % 2 == 0
    block_k = leaves * leaf
    leaf_bytes = 1024 * chunks
    a_elems, b_elems = (m - 1) * a_pitch + k, (n - 1) * b_pitch + k  # extent of each operand in elements
    groups = -(-n // COLS) * row_groups
    # the corners of the grid and a few groups in the middle
    picked = sorted({0, 1, row_groups - 1, groups - 1, groups - row_groups, groups // 2} & set(range(groups)))
    for gid, wave in itertools.product(picked, (0, NODE_WAVES - 1, 3)):
        n0, m0 = (gid // row_groups) * COLS, (gid % row_groups) * 16
        assert n0 < n and m0 < m
        wave_k = 4 * wave * block_k
        w_base, a_base = n0 * b_pitch + wave_k, m0 * a_pitch + wave_k
        for leaf_index in (0, 1, leaves - 1):
            lo = leaf_index * leaf
            seen = set()
            for j, lane in itertools.product(range(chunks), range(64)):
                g = 64 * j + lane
                pair, chunk = g // chunks, (g % chunks) ^ swizzle(g // chunks, chunks)
                col = pair & 15
                col_in = col if n0 + col < n else n - 1 - n0
                off = col_in * b_pitch + (pair >> 4) * block_k + 8 * chunk
                assert 0 <= 2 * off < 2**32
                first = w_base + lo + off
                assert 0 <= first and first + 8 <= b_elems, (m, n, k, gid, wave, leaf_index, j, lane)
                assert 1024 * j + 16 * lane + 16 <= leaf_bytes  # where the hardware puts the lane's 16 bytes
                if n0 + col < n:
                    key = (col, pair >> 4, chunk)
                    assert key not in seen
                    seen.add(key)
            assert len(seen) == min(COLS, n - n0) * 4 * chunks
            for lane in range(64):
                row = lane & 15
                row_in = row if m0 + row < m else m - 1 - m0
                off = row_in * a_pitch + (lane >> 4) * block_k
                assert 0 <= 2 * off < 2**32
                first = a_base + lo + off
                # the lane reads its leaf's chunks at off, off + 8, ...
                assert 0 <= first and first + leaf <= a_elems, (m, n, k, gid, wave, leaf_index, lane)
        # LDS: a lane's reads of both stages lie inside the wave's region, each chunk of its pair where the load put it
        for lane, c, stage in itertools.product(range(64), range(chunks), (0, 1)):
            at = lane * 16 * chunks + 16 * (c ^ swizzle(lane, chunks)) + stage * leaf_bytes
            assert at + 16 <= 2 * leaf_bytes
            g = (at - stage * leaf_bytes) // 16
            assert (g // chunks, (g % chunks) ^ swizzle(g // chunks, chunks)) == (lane, c)
    assert NODE_WAVES * 2 * leaf_bytes <= 80 * 1024  # two workgroups per CU
    assert NODE_WAVES * 2 * leaf_bytes >= NODE_WAVES * 2 * 64 * 4  # the fold's table


# up to a workgroup of 16 x 64 for every second CU (the picker's own), and grids beyond
SHAPES = [
    (1, 64, 2048), (1, 6144, 4096), (16, 100, 1536), (17, 257, 4096), (50, 64, 6144), (64, 130, 12288),
    (200, 96, 32768), (33, 320, 2048), (40, 1000, 4096), (16, 8192, 2048), (33, 2731, 6144), (8, 8190, 3072),
    (5, 4096, 4096), (32, 4096, 12288), (1000, 16, 1536), (333, 320, 24576), (64, 4096, 12288),
]  # fmt: skip


@pytest.mark.parametrize("shape", SHAPES)
def test_every_lane_address_lies_inside_its_operand(shape):
    m, n, k = shape
    model(m, n, k, k, k)
    model(m, n, k, k + 64, k + 8)  # rows that are views into wider storage


def test_which_kernel_takes_which_tree():
    assert choice(16, 64, 256) is None  # a tree of three levels
    assert choice(16, 64, 4000) is None  # ragged leaves
    assert choice(16, 64, 65536) is None  # eleven levels
    assert choice(16, 64, 512) == "rows32" and choice(16, 64, 1024) == "rows16"  # four and five levels
    assert choice(16, 4096, 12288) == "nodes" and choice(64, 4096, 12288) == "rows16" and choice(509, 6144, 4096) == "rows32"
    assert choice(32, 4096, 4096) == "nodes" and choice(33, 4096, 4096) == "rows16"  # one workgroup for every second CU
