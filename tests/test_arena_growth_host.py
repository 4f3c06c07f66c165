"""The sizes that the one-pass arena growth takes in one launch: the package's rule refuses what the
library refuses (fill and copy then grow the arena), and takes arenas of any size up to there."""
import ctypes

import pytest


@pytest.mark.parametrize("planes,slots,heads,block_bytes", [
    (56, 37450, 8, 512),                    # tiny blocks, one workgroup each: 2^24 of them
    (2, 1 << 20, 8, 16),
    (1, 1, 1 << 24, 16 << 10),
    (2, 4, 4, 8 << 30),                     # 2^24 workgroups of large blocks: 256 GiB
    (1, 1, 1, 1 << 35)])                    # a block of 2^31 vectors
def test_refused_sizes(pkg, planes, slots, heads, block_bytes):
    aligned = ctypes.c_void_p(1 << 20)  # refused before anything is launched
    assert pkg.library().q3t_grow_arena(aligned, aligned, planes, slots, slots, heads, 16, block_bytes, None) == -2
    assert not pkg.packed_kv.grow_launch_fits(planes * slots * heads, block_bytes)


@pytest.mark.parametrize("blocks,block_bytes", [
    (1, 16), ((1 << 24) - 1, 16), ((1 << 24) - 1, 16 << 10), (32, 1 << 30), (64, 2 << 30), (31, 8 << 30)])
def test_taken_sizes(pkg, blocks, block_bytes):
    assert pkg.packed_kv.grow_launch_fits(blocks, block_bytes)
