"""The kernels with a lane per ray against the oracle, on the batches that the default launch
shape would give four lanes per ray: the record-layout tests of test_gpu_multiscene and the
distance types again, with trace_relaid_kernel alone and with trace_fast_kernel's 1024-thread
workgroups before it, and the general march on every depth of split planes that
trace_relaid_kernel stages."""

from __future__ import annotations

import numpy as np
import pytest

from tests import test_gpu_multiscene
from tests.test_gpu_distance_dtypes import (  # noqa: F401
    test_dropin_reduced_distances, test_reduced_distances_every_store_site)
from tests.test_gpu_multiscene import (  # noqa: F401
    corpus, test_bad_child_index_at_the_descent_limit, test_known_answers_both_kernels, test_multiscene_parity,
    test_relaid_descent_limit_chains, test_relaid_env_order_entries_out_of_range_are_skipped,
    test_relaid_every_table_depth, test_relaid_exhaustive_fp16_inline_leaves,
    test_relaid_fast_and_general_launches_interleaved, test_relaid_huge_domains, test_relaid_malformed_dags,
    test_relaid_many_scenes_and_narrow_domains, test_relaid_non_finite_and_extreme_rays,
    test_relaid_random_rays_and_short_budgets, test_relaid_random_scene_counts_and_depths,
    test_relaid_randomized_sweep, test_relaid_signed_zero_axes_and_long_ranges, test_relaid_tables_below_the_planes,
    test_unknown_scene_id_reports_nan)

pytestmark = pytest.mark.gpu

_run = test_gpu_multiscene._run


@pytest.fixture(autouse=True, params=["combined", "wide"])
def lanes(gpu, request, monkeypatch):
    """The launch shape, and a look at every launch of a test's ``_run``: trace_relaid_kernel
    is enqueued, with trace_fast_kernel's wide workgroups before it or alone."""
    from navi_amd import _native

    wide = request.param == "wide"

    def run(*args, **kw):
        got = _run(*args, **kw)
        info = _native.last_launch()
        assert info["raw"] or (info["combined"] and not info["quad"] and (wide or not info["fast"])), info
        return got

    monkeypatch.setattr(test_gpu_multiscene, "_run", run)
    prev = _native.set_wide_min_rays(0 if wide else (1 << 64) - 1)
    yield run
    _native.set_wide_min_rays(prev)


# (table depth, plane depth): the instances of trace_relaid_kernel, without planes at depths 5 and 6
INSTANCES = [(4, 4), (5, 4), (6, 4), (5, 5), (6, 5), (7, 5), (6, 6), (7, 6), (5, 0), (6, 0)]


@pytest.mark.parametrize("negative", [False, True])
@pytest.mark.parametrize("depth,planes", INSTANCES)
def test_general_march_on_every_plane_depth(lanes, corpus, depth, planes, negative):  # noqa: F811
    """A range of 1200 m over monotone scenes, and scenes with a negative leaf (which keep
    the void cache): canonical rays and random ones from in and around the domains."""
    from navi_amd import _native
    from navi_amd.multiscene import ResidentScenes, plane_depth

    n = next(n for n in range(1, 400) if plane_depth(n, depth) == planes)
    words = [c.words for c in corpus]
    if negative:
        words[1] = words[1].copy()
        leaf = np.flatnonzero(words[1] >> np.uint64(63))
        words[1][leaf[:: leaf.size // 7]] |= np.uint64(0x8000)
        n += n == 1  # (a pool of the first scene alone has none)
        assert plane_depth(n, depth) == planes
    many = [(words[i % 4], corpus[i % 4].bbox_min_list, corpus[i % 4].bbox_max) for i in range(n)]
    bounds = [list(s[1]) + list(s[2]) for s in many]
    res = ResidentScenes(many, table_depth=depth)
    max_distance = 30.0 if negative else 1200.0
    env_scene, o, d = test_gpu_multiscene._rays(corpus, 20, 16, 16, seed=depth + planes)
    env_scene = (env_scene + 4 * np.arange(20, dtype=np.int32)) % n
    rng = np.random.default_rng(depth * 8 + planes)
    lo = np.array([bounds[s][:3] for s in env_scene]) - 2.0
    hi = np.array([bounds[s][3:] for s in env_scene]) + 2.0
    o2 = rng.uniform(lo[:, None, :], hi[:, None, :], (20, 256, 3))
    d2 = rng.normal(size=(20, 256, 3))
    d2[:, :20, 0] = 0.0  # some parallel to the x planes
    d2 /= np.linalg.norm(d2, axis=-1, keepdims=True)
    for rays, bins in (((o, d), 16), ((o2.astype(np.float32), d2.astype(np.float32)), None)):
        ref = test_gpu_multiscene._oracle_multi([s[0] for s in many], bounds, env_scene, *rays, 200, max_distance)
        got = lanes(res, env_scene, *rays, 200, max_distance, elevation_bins=bins)
        assert _native.last_launch()["planes"] == planes
        test_gpu_multiscene._compare(got, ref, max_distance, f"{planes}/{depth}/{negative}/{bins}")
