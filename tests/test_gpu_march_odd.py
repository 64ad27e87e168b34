"""The traversal loop for well-behaved rays and the general one behind it (march_step): rays and
octrees at the line between the two, against the oracle, on every schedule.

Reference: shader/octree.glsl:47-177,179-340,342-629.  Records are bit-exact, so no tolerance.
"""
import math

import numpy as np
import pytest

import oracle
from svo_testutil import hits_equal

pytestmark = pytest.mark.gpu

LEAF, NODE = 0xC1000000, 0x80000000


def deep_chain(depth, fan):
    """Blocks 0..depth-1: `fan` children of every block point to the next one (the last block's are
    leaves), the others are empty."""
    w = np.zeros(8 * depth, np.uint32)
    for d in range(depth):
        for c in fan:
            w[8 * d + c] = LEAF | (0x010203 * (d + 1) & 0xFFFFFF) if d == depth - 1 else NODE | 8 * (d + 1)
    return w


def scene_words(ctx, level=6):
    import sparsevoxeloctree_amd as S

    xyz, rgb = S.gen_scene(1, 0x0DD, 6)
    sc = S.Scene.Create(ctx, xyz, rgb)
    vox = S.Voxelizer.Create(sc, level)
    vox.CmdVoxelize()
    b = S.OctreeBuilder.Create(vox)
    b.CmdBuild()
    return b.GetOctree().words()


def octree_case(ctx, name):
    if name == "scene":
        return scene_words(ctx), 6
    if name == "one_block":  # W = 8, the smallest octree
        return np.array([0, LEAF | 7, 0, 0, LEAF | 9, 0, 0, LEAF], np.uint32), 1
    if name == "no_flag":  # non-zero words without the non-empty bit: the march keeps such a word
        w = scene_words(ctx).copy()
        leaf = np.nonzero(w >> 30 == 3)[0][::7]
        w[leaf] &= 0x7FFFFFFF
        return w, 6
    if name == "depth_12":
        return deep_chain(12, (0, 3, 5, 6)), 12
    return deep_chain(13, (0, 3, 5, 6)), 12  # a leaf one level below the deepest legal one


def odd_rays(seed, n):
    rng = np.random.default_rng(seed)
    o = rng.uniform(1.0, 2.0, (n, 3))
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    q = n // 8
    o[:q] = rng.uniform(-3.0, 6.0, (q, 3))  # most of these miss the cube
    d[q:2 * q] *= 2.0 ** rng.integers(-60, 60, (q, 1))  # unnormalised
    d[2 * q:3 * q] *= 10.0 ** rng.uniform(-30, 0, (q, 3))  # components below the EPS clamp
    o[3 * q:4 * q] = 1.5 - d[3 * q:4 * q] * 10.0 ** rng.uniform(0, 1.5, (q, 1))  # far origins, aimed at the cube
    d[4 * q:5 * q] *= 2.0 ** 90.0  # t_coef too small for the fast loop
    o[5 * q:6 * q] = np.round(o[5 * q:6 * q] * 64) / 64  # through cell corners
    d[5 * q:6 * q] = np.sign(d[5 * q:6 * q]) / math.sqrt(3.0)
    d[6 * q:7 * q, rng.integers(0, 3)] = 0.0
    return np.concatenate([o, d], axis=1).astype(np.float32)


def march_all(ctx, octree, rays, variant):
    """Records of every schedule of svo_march_rays and of the batch entry point."""
    import sparsevoxeloctree_amd as S
    from sparsevoxeloctree_amd._capi import lib

    out = []
    for mode in (0, 1):
        ctx.check(lib.svo_march_mode(ctx.h, mode))
        try:
            out.append(S.march_rays(ctx, octree, rays, variant))
            cut = len(rays) // 3
            out.append(np.concatenate(S.march_rays_batch([octree, octree], [rays[:cut], rays[cut:]], variant)))
        finally:
            ctx.check(lib.svo_march_mode(ctx.h, -1))
    return out


@pytest.mark.parametrize("name", ["scene", "one_block", "no_flag", "depth_12", "depth_13"])
@pytest.mark.parametrize("variant", [0, 1, 2])
def test_odd_rays_and_octrees_match_oracle(ctx, no_device_errors, name, variant):
    import sparsevoxeloctree_amd as S

    words, level = octree_case(ctx, name)
    rays = odd_rays(5 + variant, 4001)
    oracle.reset_counters()
    ref = oracle.march_rays(words, level, rays, variant)
    assert oracle.stack_uninit_reads() == 0
    print("odd rays", name, variant, flush=True)
    octree = S.Octree.FromWords(ctx, words, level)
    for got in march_all(ctx, octree, rays, variant):
        ok, msg = hits_equal(got, ref)
        assert ok, msg


@pytest.mark.parametrize("name", ["one_block", "no_flag", "depth_13"])
def test_odd_octree_frames_match_oracle(ctx, no_device_errors, name):
    import sparsevoxeloctree_amd as S
    from sparsevoxeloctree_amd._capi import lib

    words, level = octree_case(ctx, name)
    octree = S.Octree.FromWords(ctx, words, level)
    cam = S.camera_look_at((2.6, 2.2, 0.7), (1.5, 1.5, 1.5), aspect=1.3)
    W, H = 91, 70
    beam, _ = oracle.beam(words, level, cam.uniform_array(), W, H)
    ref = oracle.march_frame(words, level, cam.uniform_array(), W, H, beam)
    print("odd frame", name, flush=True)
    for mode in (0, 1, 2):
        ctx.check(lib.svo_march_mode(ctx.h, mode))
        try:
            t = S.OctreeTracer.Create(octree, cam)
            t.Resize(W, H)
            t.CmdDrawPipeline()
            assert np.array_equal(t.GetBeam().view(np.uint32), beam.view(np.uint32))
            ok, msg = hits_equal(t.GetHits(), ref)
        finally:
            ctx.check(lib.svo_march_mode(ctx.h, -1))
        assert ok, msg
    plan_hits = S.march_batch([octree], [cam], W, H)
    ok, msg = hits_equal(plan_hits[0], ref)
    assert ok, msg


@pytest.mark.parametrize("words,bit", [
    (np.array([0, NODE | 8, 0, 0, NODE | 1000000, 0, 0, NODE | 4] + [LEAF] * 8, np.uint32), 2),  # child block past W
    (deep_chain(14, (0, 1, 2, 3, 4, 5, 6, 7)), 4),  # deeper than the stack
])
def test_malformed_octrees_raise_error_bits(ctx, words, bit):
    import sparsevoxeloctree_amd as S

    ctx.device_errors()
    octree = S.Octree.FromWords(ctx, words, 12)
    rays = odd_rays(3, 1000)
    rays = rays[np.all(np.abs(rays) < 10, axis=1)]
    print("malformed octree, bit", bit, flush=True)
    got = march_all(ctx, octree, rays, 0)
    assert ctx.device_errors() & bit
    for other in got[1:]:
        ok, msg = hits_equal(other, got[0])
        assert ok, msg


@pytest.mark.parametrize("W,H", [(8, 8), (176, 184), (184, 184), (256, 128), (203, 331), (520, 505)])
def test_frame_tiles_cover_every_pixel(ctx, no_device_errors, W, H):
    # tile counts below, at and above whole rounds of the dealing to the XCDs (512 one-wave tiles,
    # 128 16x16 tiles), with partial tiles, in every one-ray-per-lane schedule
    import sparsevoxeloctree_amd as S
    from sparsevoxeloctree_amd._capi import lib, ptr

    blank = np.zeros(3 * W * H * 8, np.uint32)
    words = scene_words(ctx)
    octree = S.Octree.FromWords(ctx, words, 6)
    cam = S.camera_look_at((2.3, 2.0, 0.8), (1.5, 1.5, 1.5), aspect=W / H)
    beam, _ = oracle.beam(words, 6, cam.uniform_array(), W, H)
    ref = oracle.march_frame(words, 6, cam.uniform_array(), W, H, beam)
    print("frame tiles", W, H, flush=True)
    for mode in (0, 1, 2):
        ctx.check(lib.svo_march_mode(ctx.h, mode))
        try:
            t = S.OctreeTracer.Create(octree, cam)
            t.Resize(W, H)
            t._ensure()
            ctx.check(lib.svo_upload(ctx.h, t.hits.ptr, ptr(blank), W * H * 32))
            t.CmdDrawPipeline()
            ok, msg = hits_equal(t.GetHits(), ref)
        finally:
            ctx.check(lib.svo_march_mode(ctx.h, -1))
        assert ok, "mode %d: %s" % (mode, msg)
    for shape in (0, 1, 2, 3):
        plan = S.MarchPlan([octree] * 3, [cam] * 3, W, H)
        plan.set_shape(shape)
        hits = plan.alloc_hits()
        ctx.check(lib.svo_upload(ctx.h, hits.ptr, ptr(blank), 3 * W * H * 32))
        plan.run(hits)
        got = hits.download(S.HIT_DTYPE, 3 * W * H).reshape(3, H, W)
        for k in range(3):
            ok, msg = hits_equal(got[k], ref)
            assert ok, "shape %d frame %d: %s" % (shape, k, msg)


@pytest.mark.parametrize("R", [1, 65, 1023, 1025, 66567])
def test_ray_pool_sizes_match_oracle(ctx, no_device_errors, R):
    # whole and partial pools of the refill schedule (1024 rays), around its dealing to the XCDs (64 pools)
    import sparsevoxeloctree_amd as S

    words = scene_words(ctx)
    octree = S.Octree.FromWords(ctx, words, 6)
    rays = odd_rays(R, max(R, 8))[:R]
    ref = oracle.march_rays(words, 6, rays, 0)
    print("ray pool", R, flush=True)
    for k, got in enumerate(march_all(ctx, octree, rays, 0)):
        ok, msg = hits_equal(got, ref)
        assert ok, "form %d: %s" % (k, msg)


@pytest.mark.parametrize("power", [60, 61, 100, 111, 112, 113, 120, -112, -149])
@pytest.mark.parametrize("variant", [0, 1, 2])
def test_direction_lengths_match_oracle(ctx, no_device_errors, power, variant):
    # directions of length 2^power: from 2^112 on the reciprocals are too small for the fast loop
    import sparsevoxeloctree_amd as S

    words = scene_words(ctx)
    octree = S.Octree.FromWords(ctx, words, 6)
    rng = np.random.default_rng(200 + power)
    o = rng.uniform(0.5, 2.5, (2000, 3))
    d = rng.normal(size=(2000, 3))
    d *= 2.0 ** (power + rng.integers(0, 2, (2000, 1))) / np.linalg.norm(d, axis=1, keepdims=True)
    rays = np.concatenate([o, d], axis=1).astype(np.float32)
    ref = oracle.march_rays(words, 6, rays, variant)
    print("direction lengths", power, variant, flush=True)
    for k, got in enumerate(march_all(ctx, octree, rays, variant)):
        ok, msg = hits_equal(got, ref)
        assert ok, "form %d: %s" % (k, msg)


@pytest.mark.parametrize("R", [262144, 262145, 600001, 1000003])
def test_ray_pool_grows_with_the_rays(ctx, no_device_errors, R):
    # pools of 256 rays up to 4 blocks per CU, then of 512, 768 and 1024: against one ray per lane, with
    # rays for the general loop among them
    import sparsevoxeloctree_amd as S

    octree = S.Octree.FromWords(ctx, scene_words(ctx), 6)
    some = odd_rays(R, 8192)
    rays = np.ascontiguousarray(some[np.random.default_rng(R).integers(0, len(some), R)])
    print("ray pool growth", R, flush=True)
    one, one_batch, pool, pool_batch = march_all(ctx, octree, rays, 0)
    for got in (one_batch, pool, pool_batch):
        ok, msg = hits_equal(got, one)
        assert ok, msg
