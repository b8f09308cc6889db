"""The one-pass direction check (navi_check_directions) against the exact checks: it accepts
only what both of them accept, whatever the batch's size, and calls next to the tolerance or
with bad directions end as the exact checks decide."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _unit(n, seed=0):
    d = np.random.default_rng(seed).normal(size=(1, n, 3))
    return (d / np.linalg.norm(d, axis=2, keepdims=True)).astype(np.float32)


# around one workgroup's 256 rays, one more than 256 workgroups take in a round, and less than a wave
@pytest.mark.parametrize("n", [1, 63, 255, 256, 257, 65536, 65537, 200_001])
def test_every_ray_is_looked_at(gpu, n):
    import torch

    from navi_amd import torch_sdf_backend as native
    from navi_amd.torch_sdf import backend

    good = _unit(n)
    dirs = torch.from_numpy(good).to("cuda")
    assert native.directions_within_tolerance(dirs) and backend._validate_direction_norms(dirs)
    for at in {0, n // 2, n - 1}:
        for bad, message in ((np.nan, "finite"), (np.inf, "finite"), (2.0, "normalized within tolerance")):
            d = good.copy()
            d[0, at, at % 3] = bad
            t = torch.from_numpy(d).to("cuda")
            assert not native.directions_within_tolerance(t)
            for check in (native._validate_direction_norms, backend._validate_direction_norms):
                with pytest.raises(RuntimeError, match=message):
                    check(t)


def test_near_the_tolerance_the_exact_checks_decide(gpu):
    """Axis-parallel directions are their own norms: 1 + 1e-4 within an ulp of binary32 is
    where the exact checks turn, inside the margin that the quick check leaves to them."""
    import torch

    from navi_amd import torch_sdf_backend as native

    edge = np.float32(1.0 + 1e-4)
    for k in range(-40, 41):
        length = edge + np.float32(k * 2.0 ** -23)
        t = torch.tensor([[[0.0, float(length), 0.0]]], device="cuda")
        assert not native.directions_within_tolerance(t) or float(length) - 1.0 <= 1e-4 - 1e-6
        if abs(float(length) - 1.0) > 1e-4:
            with pytest.raises(RuntimeError, match="normalized within tolerance"):
                native._validate_direction_norms(t)
        else:
            native._validate_direction_norms(t)


def test_other_tensors_are_left_to_the_exact_checks(gpu):
    import torch

    from navi_amd import torch_sdf_backend as native

    d = torch.from_numpy(_unit(8)).to("cuda")
    for t in (d.cpu(), d.double(), d.half(), d[:, ::2], d[:, :0], d[..., :2].contiguous()):
        assert not native.directions_within_tolerance(t)
