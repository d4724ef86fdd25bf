"""The step loop of the traversal where it can go wrong, bit for bit against
the oracle: the smallest and the largest grids, bundles of rays whose waves
enter their first levels together, waves that mix octants, rays along axes,
from far away and with infinite or undefined numbers, and the bound on the
number of cells a walk looks up."""
import numpy as np
import pytest

import oracle_py as O
from scenes import random_points

pytestmark = pytest.mark.gpu


def _check(log2, pts, rays, flags=0):
    from pyrit_amd import gpu

    b = gpu.build(log2, pts)
    got = gpu.trace_dag(b.dag(), rays, flags)
    want = O.trace_dag_rays(O.build_points(log2, pts), rays, flags)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    return want


def _rays(origins, directions, tmin=0.0, tmax=3.402823466e38):
    from pyrit_amd import abi

    r = np.zeros(len(origins), abi.RAY)
    r["origin"], r["direction"], r["tmin"], r["tmax"] = origins, directions, tmin, tmax
    return r


def _points(log2, rng):
    n = 1 << log2
    count = min(20000, n ** 3 // 3)
    pts = random_points(count, log2, seed=log2)
    if log2 > 6:  # something to hit: a slab of voxels in the middle, and its neighbours
        s = np.zeros(20000, pts.dtype)
        s["x"], s["z"] = rng.integers(n // 2 - 80, n // 2 + 80, (2, 20000))
        s["y"] = n // 2 + rng.integers(-4, 5, 20000)
        s["attribute"] = rng.integers(1, 1 << 31, 20000)
        pts = np.concatenate([pts, s])
    return pts


@pytest.mark.parametrize("log2", [3, 4, 6, 9, 12, 13, 20])
def test_ray_forms(hip_device, log2):
    rng = np.random.default_rng(log2)
    n = float(1 << log2)
    pts = _points(log2, rng)
    parts = []
    span = min(n, 200.0)
    for k in range(48):  # 64 rays from one place (inside and outside the grid) into a narrow cone
        o = n / 2 + rng.uniform(-1, 1, 3) * (span if k % 2 else n)
        d = (n / 2 + rng.uniform(-0.25, 0.25, 3) * span) - o
        parts.append(_rays(np.repeat(o[None], 64, 0), d + rng.normal(0, 0.02, (64, 3)) * np.abs(d).max()))
    o = n / 2 + rng.uniform(-1, 1, (4096, 3)) * span
    parts.append(_rays(o, rng.normal(0, 1, (4096, 3))))
    axis = np.eye(3)[rng.integers(0, 3, 2048)] * rng.choice([-1.0, 1.0], (2048, 1))
    parts.append(_rays(n / 2 + rng.uniform(-1, 1, (2048, 3)) * span, axis))
    parts.append(_rays(np.floor(n / 2 + rng.uniform(-1, 1, (1024, 3)) * span), np.sign(rng.normal(0, 1, (1024, 3)))))
    d = rng.normal(0, 1, (1024, 3))
    parts.append(_rays(n / 2 - d * 1e7, d))
    parts.append(_rays(n / 2 - d * 1e9, d, tmin=1e8))
    parts.append(_rays(o[:1023], rng.normal(0, 1, (1023, 3)), tmin=span / 8, tmax=span / 2))
    odd = _rays(o[:1024], rng.normal(0, 1, (1024, 3)))
    for i, value in enumerate([np.inf, -np.inf, np.nan, 0.0, -0.0, 1e-38, 1e38]):
        odd["direction"][i::16, i % 3] = value
        odd["origin"][i + 8::16, i % 3] = value
    parts.append(odd)
    want = _check(log2, pts, np.concatenate(parts))
    assert (want["instance"] == 0).sum() > 500


def test_lookup_bound(hip_device):
    # a row of voxels under the ray keeps it at single voxels; the walk gives
    # up after 65536 lookups, which lies between the nearest and farthest start
    log2, n = 17, 1 << 17
    from pyrit_amd import abi

    pts = np.zeros(n + 1, abi.VOXEL)
    pts["x"][:n] = np.arange(n)
    pts["x"][n], pts["y"][n] = n - 1, 1
    pts["attribute"] = 7
    start = n - 1 - np.arange(15000, 66000, 7)
    o = np.stack([start + 0.5, np.full(len(start), 1.5), np.full(len(start), 0.5)], 1)
    want = _check(log2, pts, _rays(o, np.tile([1.0, 0.0, 0.0], (len(start), 1))))
    found = want["instance"] == 0
    assert found.any() and not found.all()
