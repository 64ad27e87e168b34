"""Small batches take fewer launches: scans of one block with the steps around them, tables as kernel
arguments, descriptors written to the host by the kernel.  Sizes around each line, against the oracle;
fragment lists and words are exact, so no tolerance.

Reference: src/Voxelizer.cpp:134-179, src/OctreeBuilder.cpp:142-214.
"""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def triangles(n, seed):
    rng = np.random.default_rng(seed)
    a = rng.uniform(-0.9, 0.9, (n, 1, 3))
    xyz = (a + rng.uniform(-0.05, 0.05, (n, 3, 3))).astype(np.float32)
    return xyz.reshape(n, 9), rng.integers(0, 1 << 24, n, dtype=np.uint32)


def run(ctx, sizes, levels):
    import sparsevoxeloctree_amd as S

    inputs = [triangles(n, 7 * i + n) for i, n in enumerate(sizes)]
    scenes = [S.Scene.Create(ctx, x, c, normalize=False) for x, c in inputs]
    voxs = S.voxelize_batch(scenes, levels)
    octs = S.build_batch(voxs)
    for (x, c), lv, v, o in zip(inputs, levels, voxs, octs):
        ref = oracle.voxelize(x, c, lv)
        assert np.array_equal(v.GetVoxelFragmentList(), ref)
        assert np.array_equal(o.words(), oracle.build(ref, lv))


# triangles: one block scans up to 4096 counts; levels 7 and 8: 1,170 and 9,363 rank chunks
@pytest.mark.parametrize("n", [1, 2, 4095, 4096, 4097])
@pytest.mark.parametrize("level", [1, 2, 6, 7, 8])
def test_one_scene(ctx, n, level):
    print("one", n, level, flush=True)
    run(ctx, [n], [level])


# scenes: one, tables above 1 KB from a few scenes on, 64 and 65 around the kernel-written read-back
@pytest.mark.parametrize("scenes", [2, 3, 4, 64, 65])
@pytest.mark.parametrize("top", [5, 8])
def test_batches(ctx, scenes, top):
    print("batch", scenes, top, flush=True)
    run(ctx, [1 + (37 * i) % 90 for i in range(scenes)], [1 + i % top for i in range(scenes)])


# leaf blocks around the line of the bin scan: every second voxel of a plane has a block of its own
@pytest.mark.parametrize("blocks", [4095, 4096, 4097])
def test_bins(ctx, blocks):
    import sparsevoxeloctree_amd as S
    from svo_testutil import pack_frags

    k = np.arange(blocks)
    rng = np.random.default_rng(blocks)
    fr = pack_frags(2 * (k % 64), 2 * (k // 64 % 64), 2 * (k // 4096), rng.integers(0, 1 << 24, blocks))
    print("bins", blocks, flush=True)
    b = S.OctreeBuilder.Create(S.Voxelizer.FromFragments(ctx, fr, 7))
    b.CmdBuild()
    assert np.array_equal(b.GetOctree().words(), oracle.build(fr, 7))


def test_plan_replays(ctx):
    # the same kernels captured and replayed, with other triangles each time
    import sparsevoxeloctree_amd as S

    level, n = 6, 500
    x, c = triangles(n, 1)
    scene = S.Scene.Create(ctx, x, c, normalize=False)
    plan = S.BuildPlan([scene], [level], [200000], [1 << 18])
    for seed in (2, 3, 4, 2):
        x, c = triangles(n, seed)
        scene.update(x, c, normalize=False)
        print("plan", seed, flush=True)
        plan.run()
        plan.finish()
        ref = oracle.voxelize(x, c, level)
        assert np.array_equal(plan.fragments(0).GetVoxelFragmentList(), ref)
        assert np.array_equal(plan.octree(0).words(), oracle.build(ref, level))
