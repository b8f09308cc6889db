"""GPU parity of the small-batch tracer (trace_quad_kernel, four lanes per ray) against the
CPU oracle at the edges of its units: rays per env around 4 and 16, batches on both sides
of its 4-ray units (2^14 rays) and of the 512 units that an XCD round spans, tiled and
linear order, with its fast and its general march."""

from __future__ import annotations

import numpy as np
import pytest

from tests.test_gpu_multiscene import _compare, _oracle_multi, _rays, _run, corpus  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def resident(gpu, corpus):  # noqa: F811
    from navi_amd.multiscene import ResidentScenes

    return ResidentScenes([(c.words, c.bbox_min_list, c.bbox_max) for c in corpus])


# (envs, az, el, elevation_bins): 1 ray; 3, 15, 17 and 65 rays per env; a batch of 4-ray
# tiles; 16-ray units, one more than 512 of them and a tiled batch
SHAPES = [(1, 1, 1, 0), (5, 3, 1, 0), (7, 5, 3, 0), (3, 17, 1, 0), (2, 13, 5, 0), (4, 16, 8, 8), (30, 32, 17, 0),
          (513, 16, 2, 0), (21, 32, 32, 32)]


@pytest.mark.parametrize("max_distance", [30.0, 1200.0])
@pytest.mark.parametrize("envs,az,el,bins", SHAPES)
def test_quad_units_match_the_oracle(resident, corpus, envs, az, el, bins, max_distance):  # noqa: F811
    from navi_amd import _native

    env_scene, o, d = _rays(corpus, envs, az, el, seed=envs + az)
    if envs > 2:
        env_scene[1] = 99  # an unknown scene: NaN, semantic 0, no steps
    ref = _oracle_multi([c.words for c in corpus], [c.bbox_min_list + c.bbox_max for c in corpus],
                        np.where(env_scene == 99, 0, env_scene).astype(np.int32), o, d, 160, max_distance)
    if envs > 2:
        ref["distance"][1], ref["semantic"][1], ref["steps"][1] = np.nan, 0, 0
    got = _run(resident, env_scene, o, d, 160, max_distance, elevation_bins=bins)
    info = _native.last_launch()
    assert info["quad"] and info["n_rays"] == envs * az * el, info
    assert not (info["combined"] or info["fast"] or info["raw"]), info  # nothing else is enqueued
    _compare(got, ref, max_distance, f"{envs}x{az}x{el}/{bins}/{max_distance}")


# one wave with fewer than, exactly and more than 16 rays; envs of different scenes in one wave; several
# waves; a tiled batch
@pytest.mark.parametrize("envs,az,el,bins", SHAPES + [(1, 15, 1, 0), (1, 16, 1, 0), (16, 1, 1, 0), (33, 1, 2, 0)])
@pytest.mark.parametrize("steps", [160, 7])
def test_last_rays_of_a_wave_match_the_oracle(resident, corpus, envs, az, el, bins, steps):  # noqa: F811
    """The one-lane-per-ray kernel, whose waves hand their last 16 rays to quads: rays
    handed over before their first step, between steps, and close to the step limit."""
    from navi_amd import _native

    env_scene, o, d = _rays(corpus, envs, az, el, seed=envs + az)
    o = o.copy()
    o[0, 0] = [1e3, 1e3, 1e3]  # a ray from outside the domain
    ref = _oracle_multi([c.words for c in corpus], [c.bbox_min_list + c.bbox_max for c in corpus],
                        env_scene.astype(np.int32), o, d, steps, 30.0)
    prev = _native.set_wide_min_rays(0)
    try:
        got = _run(resident, env_scene, o, d, steps, 30.0, elevation_bins=bins)
        info = _native.last_launch()
    finally:
        _native.set_wide_min_rays(prev)
    assert info["fast_wide"] and not info["quad"] and info["fast_planes"] == 8, info
    _compare(got, ref, 30.0, f"{envs}x{az}x{el}/{bins}/{steps}")


@pytest.mark.parametrize("envs", [103, 104, 159, 160])
def test_launch_shapes_of_mid_size_batches(resident, corpus, envs):  # noqa: F811
    """8192 rays an env on both sides of the lines between four lanes per ray and one
    (851,968 rays), and between one workgroup per CU and two whose waves thin out
    towards the end (1,310,720)."""
    from navi_amd import _native

    env_scene, o, d = _rays(corpus, envs, 128, 64, seed=envs)
    ref = _oracle_multi([c.words for c in corpus], [c.bbox_min_list + c.bbox_max for c in corpus],
                        env_scene.astype(np.int32), o, d, 160, 30.0)
    got = _run(resident, env_scene, o, d, 160, 30.0, elevation_bins=64)
    info = _native.last_launch()
    # 256 CUs of 16 or 32 waves
    assert info["quad"] == (envs < 104) and (info["quad"] or info["waves"] == (4096 if envs < 160 else 8192)), info
    _compare(got, ref, 30.0, str(envs))


# (envs, az, el, elevation_bins, max_distance, quads): units on both sides of each line. Envs of
# 3 rays (a unit each), full units of 128 rays an env (8 each), in tiles too, of 127 (one idle
# lane in 128, but an env too small for its neighbours to be alike), of 64 in tiles and of 16 (full,
# too small); angular tiles over a general range (4 units each); 16,384 envs of one ray (the
# smallest launches) and one more
LINES = [(8191, 3, 1, 0, 30.0, True), (8192, 3, 1, 0, 30.0, False), (4095, 128, 1, 0, 30.0, True),
         (4096, 128, 1, 0, 30.0, False), (1023, 127, 1, 0, 30.0, True), (1024, 127, 1, 0, 30.0, False),
         (4095, 16, 8, 8, 30.0, True), (4096, 16, 8, 8, 30.0, False), (2047, 8, 8, 8, 30.0, True),
         (2048, 8, 8, 8, 30.0, False), (8191, 16, 1, 0, 30.0, True), (8192, 16, 1, 0, 30.0, False), (1023, 8, 8, 8, 1200.0, True),
         (1024, 8, 8, 8, 1200.0, False), (16384, 1, 1, 0, 30.0, True), (16385, 1, 1, 0, 30.0, False)]


@pytest.mark.parametrize("envs,az,el,bins,max_distance,quads", LINES)
def test_launches_of_many_units_leave_the_quads(resident, corpus, envs, az, el, bins, max_distance, quads):  # noqa: F811
    from navi_amd import _native

    env_scene, o, d = _rays(corpus, envs, az, el, seed=envs + az)
    ref = _oracle_multi([c.words for c in corpus], [c.bbox_min_list + c.bbox_max for c in corpus],
                        env_scene, o, d, 96, max_distance)
    got = _run(resident, env_scene, o, d, 96, max_distance, elevation_bins=bins)
    info = _native.last_launch()
    assert info["quad"] == quads, info
    _compare(got, ref, max_distance, f"{envs}x{az}x{el}/{bins}/{max_distance}")


@pytest.mark.parametrize("envs,quads", [(1023, True), (1024, False)])
def test_launches_of_negative_leaves_leave_the_quads_early(gpu, corpus, envs, quads):  # noqa: F811
    """Scenes that need the general march: known to ResidentScenes, so their line is its."""
    from navi_amd import _native
    from navi_amd.multiscene import ResidentScenes

    words = corpus[1].words.copy()
    leaf = np.flatnonzero(words >> np.uint64(63))
    words[leaf[leaf.size // 2]] |= np.uint64(0x8000)
    bounds = corpus[1].bbox_min_list + corpus[1].bbox_max
    resident = ResidentScenes([(words, bounds[:3], bounds[3:])])
    env_scene, o, d = _rays(corpus[1:2], envs, 8, 8, seed=envs)
    ref = _oracle_multi([words], [bounds], env_scene, o, d, 96, 30.0)
    got = _run(resident, env_scene, o, d, 96, 30.0, elevation_bins=8)
    info = _native.last_launch()
    assert info["quad"] == quads, info
    _compare(got, ref, 30.0, str(envs))


@pytest.mark.parametrize("sides", [0, 30, 60, 100, 200, 254, 258, 1000])
def test_scenes_far_from_the_origin(gpu, corpus, sides):  # noqa: F811
    """Boxes up to 256 of their sides away take the quads' fast march (off <= 2^16), farther
    ones the general march; depth-8 cells are 2^8 ulps wide at that line."""
    from navi_amd import _native
    from navi_amd.multiscene import ResidentScenes

    scene = corpus[1]
    lo, hi = np.float32(scene.bbox_min_list), np.float32(scene.bbox_max)
    side = hi[0] - lo[0]
    shift = np.float32([sides, -sides, sides]) * side
    lo, hi = lo + shift, hi + shift
    resident = ResidentScenes([(scene.words, lo.tolist(), hi.tolist())])
    env_scene, o, d = _rays(corpus[1:2], 6, 32, 16, seed=sides + 1)
    rng = np.random.default_rng(sides)
    o = (o + shift).astype(np.float32)
    o[3:] = rng.uniform(lo, hi, o[3:].shape)  # any place, cell faces among them at this spacing
    ref = _oracle_multi([scene.words], [lo.tolist() + hi.tolist()], env_scene, o, d, 160, 30.0)
    got = _run(resident, env_scene, o, d, 160, 30.0, elevation_bins=16)
    assert _native.last_launch()["quad"]
    assert resident._scene_hints == (_native.SCENES_FAST if sides <= 60 else 0)
    _compare(got, ref, 30.0, f"{sides} sides away")
