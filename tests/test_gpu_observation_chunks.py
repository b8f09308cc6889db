"""The post-pass where a workgroup walks its env in chunks of azimuth bins, at both of its
workgroup sizes, and its first-frame test, against the CPU oracle (bars of
test_gpu_observation)."""

from __future__ import annotations

import numpy as np
import pytest

import oracle
from tests.test_gpu_observation import DEPTH_RTOL, _observe_oracle_check, _resident, corpus  # noqa: F401

pytestmark = pytest.mark.gpu


def _observe(res, d, az, el, sem=None, prev=None, shift=0):
    """(fp16 depth, stats, collision, obs, delta); the fp16 output `shift` halves off its alignment."""
    import torch

    dev, e = res.device, d.shape[0]
    store = torch.empty(e * az * el + shift, dtype=torch.float16, device=dev)
    d16 = store[shift:].view(e, 1, el, az)
    st, co = torch.empty((e, 5), device=dev), torch.empty((e,), dtype=torch.int32, device=dev)
    more = {}
    if sem is not None:
        more = {"semantics": torch.from_numpy(sem).to(dev), "out_obs": torch.empty((e, 3, az, el), device=dev),
                "prev_depth": torch.from_numpy(prev).to(dev), "out_delta": torch.empty((e, az, el), device=dev)}
    res.observe(torch.from_numpy(d).to(dev), az, el, 30.0, out_depth_f16=d16, out_stats=st, out_collision=co, **more)
    torch.cuda.synchronize()
    out = [t.cpu().numpy() for t in (d16, st, co)]
    return out + [more[k].cpu().numpy() for k in ("out_obs", "out_delta", "prev_depth") if k in more]


# at most 256 envs (1024 threads): 4 and 3 chunks of 128 bins; of odd and even Az not in fours (2- and
# 4-byte copy-out), El not in fours (4-byte loads); a last chunk of one bin; four-row tiles; El too
# large for any tile. Above (512 threads): 4 chunks of 24 bins, odd ones, and the direct stores.
SHAPES = [(3, 512, 96), (2, 384, 96), (2, 513, 97), (3, 302, 130), (2, 129, 384), (2, 23, 2048), (2, 8, 6000),
          (257, 80, 256), (257, 81, 255), (257, 4, 3001), (257, 1, 8), (2, 1, 4)]


@pytest.mark.parametrize("e,az,el", SHAPES)
def test_chunked_envs_match_the_oracle(gpu, corpus, e, az, el):  # noqa: F811
    res = _resident(corpus)
    rng = np.random.default_rng(az * el)
    n = az * el
    d = rng.uniform(-1.0, 40.0, (e, n)).astype(np.float32)
    d[0, : min(4, n)] = [np.inf, -np.inf, 0.0, 30.0][: min(4, n)]
    d[1, n - 1] = np.nan  # the env's last element
    sem = rng.integers(0, 40, (e, n)).astype(np.int32)
    prev = rng.uniform(0.1, 1.0, (e, az, el)).astype(np.float32)
    prev[0] = 0.0
    want = oracle.observe(d, az, el, 30.0, 1.5, 30.0, 2.0, 0.15, semantics=sem, prev_depth=prev)
    got = _observe(res, d, az, el, sem, prev)
    _observe_oracle_check(got[:3], want)
    np.testing.assert_array_equal(got[3][:, 1:], want["obs"][:, 1:])
    assert np.array_equal(np.isnan(got[3][:, 0]), np.isnan(want["obs"][:, 0]))
    np.testing.assert_allclose(np.nan_to_num(got[3][:, 0]), np.nan_to_num(want["obs"][:, 0]), rtol=DEPTH_RTOL, atol=1e-7)
    np.testing.assert_allclose(np.nan_to_num(got[4]), np.nan_to_num(want["delta"]), rtol=0, atol=DEPTH_RTOL)
    assert np.array_equal(got[5].view(np.uint32), got[3][:, 0].view(np.uint32))
    for shift in (0, 1, 2):  # the fp16 depth alone, at every alignment of its copy-out
        part = _observe(res, d, az, el, shift=shift)
        _observe_oracle_check(part, want)
        assert np.array_equal(part[1].view(np.uint32), got[1].view(np.uint32))


# envs that end below, at and past a wave's run: of 64 elements (El not in fours), of 256 (16-byte
# accesses), of a round of all 512 or 1024 threads
ENDS = [(9, 7), (32, 2), (13, 5), (63, 4), (64, 4), (65, 4), (73, 7), (128, 4), (171, 3), (1023, 4), (1024, 4),
        (1025, 4), (24, 9)]


@pytest.mark.parametrize("e", [2, 258])
@pytest.mark.parametrize("az,el", ENDS)
def test_small_envs_match_the_oracle(gpu, corpus, e, az, el):  # noqa: F811
    """Waves that hold none of their env's elements leave the round early."""
    test_chunked_envs_match_the_oracle(gpu, corpus, e, az, el)


@pytest.mark.parametrize("e", [6, 262])
def test_first_frame_is_decided_by_the_whole_row(gpu, corpus, e):  # noqa: F811
    """The delta is zero exactly where |previous depth| sums below 1e-6: rows of zeros, of
    one late value, of values that only together reach 1e-6, that stay below it, with a
    late NaN, and whose first value is enough."""
    res = _resident(corpus)
    az, el = 96, 37
    rng = np.random.default_rng(5)
    d = rng.uniform(0.2, 20.0, (e, az * el)).astype(np.float32)
    sem = np.zeros((e, az * el), np.int32)
    prev = np.zeros((e, az, el), np.float32)
    prev[1, -1, -1] = 0.25
    prev[2] = 2e-9  # 3552 values: 7.1e-6
    prev[3] = 1e-10  # 3.6e-7
    prev[4, -1, -1] = np.nan
    prev[5, 0, 0] = -0.5
    before = prev.copy()
    got = _observe(res, d, az, el, sem, prev)
    q, delta = got[3][:, 0], got[4]
    for row, first in enumerate((True, False, False, True, False, False)):
        want = np.zeros_like(q[row]) if first else q[row] - before[row]
        assert np.array_equal(delta[row].view(np.uint32), want.view(np.uint32)) or (
            row == 4 and np.isnan(delta[row]).sum() == 1
            and np.array_equal(np.nan_to_num(delta[row]), np.nan_to_num(want)))
    assert (delta[6:] == 0).all()
