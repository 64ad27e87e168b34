"""The fold of leaf blocks with 17..64 fragments, 8 per wave: sizes around the half-wave and wave lines,
list lengths around a wave's 8 and a block's 32, mixed sizes and scenes, against the oracle (words are
exact, so no tolerance).

Reference: shader/octree_tag_node.comp:43-57.
"""
import numpy as np
import pytest

import oracle
from svo_testutil import pack_frags

pytestmark = pytest.mark.gpu


def blocks_of(sizes, level, rng, raw=False):
    """One leaf block per size, fragments anywhere in it, in random order."""
    res = 1 << level
    side = res // 2
    parts = []
    for k, n in enumerate(sizes):
        b = np.array([k % side, k // side % side, k // side // side]) * 2
        p = b + rng.integers(0, 2, (n, 3))
        c = rng.integers(0, 1 << 24, n) & int(rng.choice([0xFFFFFF, 0x030303, 0]))
        parts.append(pack_frags(p[:, 0], p[:, 1], p[:, 2], c))
    if raw:  # a coordinate past the volume: the scene's keys become fragment indices
        parts.append(pack_frags([res + 5], [res - 1], [res - 1], [77]))
    fr = np.concatenate(parts)
    return np.ascontiguousarray(fr[rng.permutation(len(fr))])


def check(ctx, lists, levels):
    import sparsevoxeloctree_amd as S

    voxs = [S.Voxelizer.FromFragments(ctx, f, lv) for f, lv in zip(lists, levels)]
    for o, f, lv in zip(S.build_batch(voxs), lists, levels):
        assert np.array_equal(o.words(), oracle.build(f, lv)), lv


@pytest.mark.parametrize("raw", [False, True])
@pytest.mark.parametrize("n", [16, 17, 31, 32, 33, 63, 64, 65])
@pytest.mark.parametrize("count", [1, 7, 8, 9, 33])
def test_equal_sizes(ctx, n, count, raw):
    print("mid", n, count, raw, flush=True)
    check(ctx, [blocks_of([n] * count, 5, np.random.default_rng(100 * n + count), raw)], [5])


@pytest.mark.parametrize("count", [256, 257, 3000])
def test_mixed_sizes_and_scenes(ctx, count):
    rng = np.random.default_rng(count)
    lists = [blocks_of(rng.choice([1, 4, 16, 17, 24, 32, 33, 48, 64, 70], count), 6, rng),
             blocks_of(rng.integers(17, 65, count // 3), 5, rng, raw=True),
             blocks_of(rng.integers(15, 40, count), 7, rng)]
    print("mixed", count, flush=True)
    check(ctx, lists, [6, 5, 7])
