"""The build's fragment tiles (groups of neighbouring leaf blocks per 1024 fragments) and the two forms
of its fold keys, against the oracle; words are exact, so no tolerance.

Reference: shader/octree_tag_node.comp:18-60.
"""
import numpy as np
import pytest

import oracle
from svo_testutil import pack_frags, random_frags

pytestmark = pytest.mark.gpu


def build_words(ctx, frags, level):
    import sparsevoxeloctree_amd as S

    b = S.OctreeBuilder.Create(S.Voxelizer.FromFragments(ctx, frags, level))
    b.CmdBuild()
    return b.GetOctree().words()


def check(ctx, frags, level):
    got, ref = build_words(ctx, frags, level), oracle.build(frags, level)
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("level", [1, 2, 5, 9, 12])
@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 5000])
def test_tile_edges(ctx, level, n):
    # random coordinates: at level 9 and 12 nearly every fragment is a group of its own, far more than
    # a tile's table holds
    print("tiles", level, n, flush=True)
    check(ctx, random_frags(100 * level + n, level, n), level)


@pytest.mark.parametrize("level,extent", [(6, 4), (10, 9), (12, 200), (12, 4094)])
def test_clustered_tiles(ctx, level, extent):
    # few leaf blocks per tile, in raster-like and in shuffled order, up to the far corner of the volume
    rng = np.random.default_rng(level * extent)
    n = 9001
    base = np.minimum((1 << level) - 1 - extent, rng.integers(0, 1 << level, 3)) if extent < (1 << level) else np.zeros(3, int)
    base = np.maximum(base, 0)
    p = base + rng.integers(0, extent + 1, (n, 3))
    p[-40:] = (1 << level) - 1
    c = rng.integers(0, 1 << 24, n)
    for order in (np.lexsort((p[:, 0], p[:, 1], p[:, 2])), rng.permutation(n)):
        check(ctx, pack_frags(p[order, 0], p[order, 1], p[order, 2], c[order]), level)


@pytest.mark.parametrize("level", [1, 3, 8, 10])
@pytest.mark.parametrize("sizes", [(1, 4, 5, 8, 9, 16), (17, 64, 65, 200), (512, 513, 2048), (2049, 5000)])
@pytest.mark.parametrize("over", [0, 1, 900])
def test_fold_sizes_and_saturated_coordinates(ctx, level, sizes, over):
    # one leaf block per size; over: how far raw coordinates pass res - 1 (0: not at all; 1: voxel = res,
    # which a voxelized scene has; more: lists from the host, folded by the whole fragments)
    rng = np.random.default_rng([level, over, *sizes])
    res = 1 << level
    parts = []
    for k, n in enumerate(sizes):
        block = np.array([res - 2, (res - 2) if k % 2 else 0, res - 2 if k % 3 else 0])
        p = block + rng.integers(0, 2, (n, 3))
        if k:
            p[:, 1] = np.where(p[:, 1] < res - 2, p[:, 1] + min(2 * k, max(res - 4, 0)) // 2 * 2, p[:, 1])
        if over:
            push = rng.random((n, 3)) < 0.4
            p = np.where(push & (p == res - 1), np.minimum(p + rng.integers(1, over + 1, (n, 3)), 4095), p)
        parts.append(pack_frags(p[:, 0], p[:, 1], p[:, 2], rng.integers(0, 1 << 24, n) & rng.choice([0xFFFFFF, 0x0000FF, 3])))
    fr = np.concatenate(parts)
    print("fold", level, sizes, over, fr.shape, flush=True)
    check(ctx, np.ascontiguousarray(fr[rng.permutation(len(fr))]), level)


@pytest.mark.parametrize("level", [1, 4, 8, 12])
@pytest.mark.parametrize("sizes", [(2, 4, 5, 8, 9, 16), (17, 32, 33, 64), (65, 512, 513), (2048, 2049, 3000)])
@pytest.mark.parametrize("some", [1.0, 0.5, 0.01])
def test_bits_outside_the_packing(ctx, level, sizes, some):
    # host lists may have bits 24..27 of the second word set (on `some` of the fragments): no part of the
    # colour, but of the order in which a leaf's fragments are folded
    rng = np.random.default_rng([level, int(100 * some), *sizes])
    p = np.concatenate([np.tile(2 * rng.integers(0, (1 << level) // 2, 3), (n, 1)) for n in sizes])
    p = p + (rng.random(p.shape) < 0.3)
    fr = pack_frags(p[:, 0], p[:, 1], p[:, 2], rng.integers(0, 1 << 24, len(p)))
    plain = oracle.build(fr, level)
    fr[:, 1] |= np.where(rng.random(len(p)) < some, rng.integers(0, 16, len(p)), 0).astype(np.uint32) << 24
    if some > 0.1:
        assert not np.array_equal(oracle.build(fr, level), plain)
    print("bits", level, sizes, some, flush=True)
    check(ctx, np.ascontiguousarray(fr[rng.permutation(len(fr))]), level)


def test_batch_mixes_key_forms(ctx):
    import sparsevoxeloctree_amd as S

    rng = np.random.default_rng(4)
    lists = [random_frags(1, 7, 3000, hot=200), random_frags(2, 3, 40, extent=2000), np.zeros((0, 2), np.uint32),
             random_frags(3, 1, 700), random_frags(4, 5, 2500, extent=4095, hot=90), random_frags(5, 12, 1500)]
    levels = [7, 3, 4, 1, 5, 12]
    voxs = [S.Voxelizer.FromFragments(ctx, f, lv) for f, lv in zip(lists, levels)]
    print("batch", flush=True)
    for o, f, lv in zip(S.build_batch(voxs), lists, levels):
        assert np.array_equal(o.words(), oracle.build(f, lv)), lv
    assert rng is not None


def test_plan_with_a_scene_out_of_the_cube(ctx):
    # an unnormalised scene reaching past the cube gives raw coordinates above res; the plan's replays
    # switch between it and a scene inside
    import sparsevoxeloctree_amd as S

    xyz, rgb = S.gen_scene(1, 77, 3)
    inside = oracle.normalize(xyz)
    outside = inside.copy()
    outside.reshape(-1, 3)[:] = outside.reshape(-1, 3) * np.float32([0.8, 0.8, 2.5])
    level = 5
    scene = S.Scene.Create(ctx, inside, rgb, normalize=False)
    refs = [(x, oracle.voxelize(x, rgb, level)) for x in (inside, outside)]
    cap = max(len(f) for _, f in refs) + 16
    plan = S.BuildPlan([scene], [level], [cap], [1 << 18])
    saw_raw = False
    for x, f in refs + refs[::-1]:
        print("plan", len(f), flush=True)
        scene.update(x, rgb, normalize=False)
        plan.run()
        plan.finish()
        assert np.array_equal(plan.fragments(0).GetVoxelFragmentList(), f)
        assert np.array_equal(plan.octree(0).words(), oracle.build(f, level))
        z = (f[:, 0] >> 24) | ((f[:, 1] >> 28) << 8)
        saw_raw |= bool((z > (1 << level)).any() or ((f[:, 0] & 0xFFF) > (1 << level)).any()
                        or (((f[:, 0] >> 12) & 0xFFF) > (1 << level)).any())
    assert saw_raw
