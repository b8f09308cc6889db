"""navi_trace_relaid_noalloc, the tracer entry point that allocates nothing (its
work-queue counters live in a static device array), called through the C ABI:

* device memory in use (hipMemGetInfo, through torch.cuda.mem_get_info) is the same
  before and after two calls in a row, the second with a smaller batch (after one
  warm-up call, so that the HIP runtime has loaded the library's kernels, which it
  does on their first launch);
* the outputs of those two calls equal navi_trace_relaid's on the same inputs:
  distances, semantics and step counts bit for bit.

Both with four lanes per ray, which needs no counters, and with a lane per ray in either
launch shape, which does.

The scene pool is built here without ResidentScenes; in a fresh process the warm-up
call is also the entry point's first call on the device (no navi_device_init before
it), while in a full test run earlier tests have initialised the device already.
"""

from __future__ import annotations

import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _say(msg: str) -> None:
    print(f"[test_zz_no_alloc] {msg}", file=sys.stderr, flush=True)


def _pool(scenes, depth):
    """Record pool, scene descriptors and cell tables of several scenes (host arrays)."""
    from navi_amd import _native

    rtable = np.zeros(len(scenes), dtype=_native.RELAID_SCENE_DTYPE)
    recs, roff = [], 0
    for i, sc in enumerate(scenes):
        rec, root, _ = _native.relayout(sc.words)
        rec = rec.copy()
        rec[rec < 0x7FFFFFFD] += np.uint32(roff)
        rtable[i]["rec_offset"], rtable[i]["n_records"] = roff, rec.shape[0]
        rtable[i]["root_slot"] = root if root & 0x80000000 else roff + root
        rtable[i]["bbox_min"], rtable[i]["bbox_max"] = sc.bbox_min_list, sc.bbox_max
        recs.append(rec)
        roff += rec.shape[0]
    allrec = np.concatenate(recs)
    for i in range(len(scenes)):
        rtable[i]["max_depth"] = _native.record_depth(allrec, int(rtable[i]["root_slot"]))
    tables = np.concatenate([_native.cell_table(allrec, int(rtable[i]["root_slot"]), depth)
                             for i in range(len(scenes))])
    return allrec, rtable, tables


def test_noalloc_allocates_nothing_and_matches_navi_trace_relaid(gpu):
    _check_noalloc({"quad": True, "fast_wide": False, "queue": "none"})


@pytest.mark.parametrize("wide", [False, True])
def test_noalloc_with_a_lane_per_ray(gpu, wide):
    from navi_amd import _native

    prev = _native.set_wide_min_rays(0 if wide else (1 << 64) - 1)
    try:
        _check_noalloc({"quad": False, "fast_wide": wide, "queue": "scratch"})
    finally:
        _native.set_wide_min_rays(prev)


def _check_noalloc(shape):
    import torch

    from navi_amd import _native
    from navi_amd import scenes as S

    scenes = [S.rooms(seed=3, resolution=128), S.cluttered(seed=2, resolution=128)]
    for sc in scenes:
        sc.compile()
    depth = 6
    allrec, rtable, tables = _pool(scenes, depth)
    dev = torch.device("cuda:0")
    records = torch.from_numpy(allrec.view(np.int32).reshape(-1).copy()).to(dev)
    table = torch.from_numpy(rtable.view(np.uint8).copy()).to(dev)
    cells = torch.from_numpy(tables.view(np.int64)).to(dev)
    lib = _native.lib()
    rng = np.random.default_rng(17)

    # every input and output of both calls and both entry points, allocated up front
    calls = []
    for E, az, el in ((12, 64, 16), (3, 32, 8)):
        R = az * el
        env_scene = rng.integers(0, len(scenes), E).astype(np.int32)
        origins_env = np.concatenate([scenes[s].free_origins(rng, 1) for s in env_scene])
        dirs = S.world_directions(S.canonical_directions(az, el), rng.uniform(0, 2 * np.pi, E))
        origins = np.ascontiguousarray(np.broadcast_to(origins_env[:, None, :], dirs.shape))
        c = {"E": E, "R": R, "el": el, "es": torch.from_numpy(env_scene).to(dev),
             "o": torch.from_numpy(origins).to(dev), "d": torch.from_numpy(dirs).to(dev)}
        for name in ("navi_trace_relaid_noalloc", "navi_trace_relaid"):
            c[name] = (torch.full((E, R), float("nan"), device=dev),
                       torch.full((E, R), -7, device=dev, dtype=torch.int32),
                       torch.full((E, R), -7, device=dev, dtype=torch.int32))
        calls.append(c)
    stream = torch.cuda.current_stream(dev).cuda_stream

    def call(name: str, k: int) -> None:
        c = calls[k]
        od, os_, on = c[name]
        _say(f"call {k}: {name}, {c['E']} envs x {c['R']} rays")
        code = getattr(lib, name)(
            records.data_ptr(), allrec.shape[0], table.data_ptr(), len(scenes), cells.data_ptr(), depth,
            c["es"].data_ptr(), None, c["E"], c["R"], c["el"], c["o"].data_ptr(), c["d"].data_ptr(),
            od.data_ptr(), os_.data_ptr(), 128, 30.0, 0.01, on.data_ptr(), stream)
        _native.check(code)
        info = _native.last_launch()
        queue = "stream" if name == "navi_trace_relaid" and not shape["quad"] else shape["queue"]
        assert {k: info[k] for k in shape} == dict(shape, queue=queue), info

    call("navi_trace_relaid_noalloc", 1)  # warm-up: the runtime loads the kernels on first launch
    torch.cuda.synchronize()
    free_before, _ = torch.cuda.mem_get_info(dev)
    call("navi_trace_relaid_noalloc", 0)
    call("navi_trace_relaid_noalloc", 1)  # the second call of the pair, a smaller batch
    torch.cuda.synchronize()
    free_after, _ = torch.cuda.mem_get_info(dev)
    assert free_after == free_before, f"device memory in use changed by {free_before - free_after} bytes"

    for k in range(2):
        call("navi_trace_relaid", k)
    torch.cuda.synchronize()
    for k, c in enumerate(calls):
        got = [t.cpu().numpy() for t in c["navi_trace_relaid_noalloc"]]
        want = [t.cpu().numpy() for t in c["navi_trace_relaid"]]
        assert np.array_equal(got[0].view(np.uint32), want[0].view(np.uint32)), f"call {k}: distances"
        assert np.array_equal(got[1], want[1]), f"call {k}: semantics"
        assert np.array_equal(got[2], want[2]), f"call {k}: step counts"
        assert (want[2] > 0).all() and not np.isnan(want[0]).any()  # every ray traced and written
