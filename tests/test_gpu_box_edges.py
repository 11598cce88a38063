"""Rays at the edges of boxes, where one rounding of a node test decides between
a hit and a miss: every layout of the fast traversal makes the same decision
(the quantized boxes may only add hits), and none loses a hit of the reference
tree, whose single-triangle leaves are the tightest boxes."""

import numpy as np
import pytest

from rendiation_amd.acceleration import TRAVERSAL_FAST, TRAVERSAL_REFERENCE
from tests.parity import MISS, TIE_REL
from tests.test_gpu_wave_traversal import SHAPES, _say, _system, _trace

pytestmark = pytest.mark.gpu

CELLS = 16


def _grid():
    """CELLS x CELLS squares over [1, 2]^2 at z = 5, two triangles each."""
    a = 1.0 + np.arange(CELLS + 1) / CELLS
    x, y = np.meshgrid(a, a, indexing="ij")
    pos = np.stack([x, y, np.full_like(x, 5.0)], axis=2).reshape(-1, 3).astype(np.float32)
    i, j = (v.reshape(-1) for v in np.meshgrid(np.arange(CELLS), np.arange(CELLS), indexing="ij"))
    c = i * (CELLS + 1) + j
    idx = np.stack([c, c + CELLS + 1, c + CELLS + 2, c, c + CELLS + 2, c + 1], axis=1)
    return pos, idx.reshape(-1).astype(np.uint32)


def _edge_points(rng, n):
    p = 1.0 + rng.random((n, 2))
    snap = rng.integers(1, 4, n)[:, None] & np.array([1, 2])  # on lines of x, of y, or of both
    p = np.where(snap != 0, np.round(p * CELLS) / CELLS, p)
    return np.concatenate([p, np.full((n, 1), 5.0)], axis=1)


def _rays(origin, direction, tmax=np.inf):
    r = np.zeros((len(origin), 8), np.float32)
    r[:, 0:3], r[:, 4:7], r[:, 7] = origin, direction, tmax
    return r


def _check(s, rays, what):
    ref = _trace(s, rays, TRAVERSAL_REFERENCE)
    pairs = None
    for shape in SHAPES:
        _say(f"{what} {shape} n={len(rays)}")
        s.set_tune(*shape)
        got = _trace(s, rays, TRAVERSAL_FAST)
        hit = got[:, 0] != MISS
        assert not np.any((ref[:, 0] != MISS) & ~hit), (what, shape)
        if pairs is None:
            pairs = got
        was = pairs[:, 0] != MISS
        assert np.array_equal(hit, was) or (shape[5] == 2 and not np.any(was & ~hit)), (
            what, shape, int(np.sum(hit & ~was)), int(np.sum(was & ~hit)))
        t, u = (v.view(np.float32)[:, 1][was] for v in (got.copy(), pairs.copy()))
        assert np.all(np.abs(t - u) <= TIE_REL * np.abs(u)) or (shape[5] == 2 and np.all(t <= u * (1 + TIE_REL)))
    return pairs


@pytest.fixture(scope="module")
def scenes(device):
    made = {"one": _system([_grid()], blas_bin_size=1)}
    many = []
    for k in range(9):  # TLAS nodes of every width
        m = np.eye(4)
        m[0, 3], m[1, 3] = (k % 3) - 1.0, (k // 3) - 1.0
        many.append(m)
    made["instances"] = _system([_grid()], many, blas_bin_size=1, tlas_bin_size=1)
    yield made
    for s in made.values():
        s.close()


@pytest.mark.parametrize("size", [0.0, 1e-6, 1e-3, 0.25, 2.0])
@pytest.mark.parametrize("scene", ["one", "instances"])
def test_edge_aimed_rays(scenes, scene, size):
    rng = np.random.default_rng(17)
    n = 60_000
    at = _edge_points(rng, n)
    if scene == "instances":
        at[:, 0:2] += rng.integers(-1, 2, (n, 2))
    origin = (rng.uniform(-1, 1, (n, 3)) * size).astype(np.float32)
    pairs = _check(scenes[scene], _rays(origin, at - origin), f"edges {scene} {size}")
    assert 0.5 < np.mean(pairs[:, 0] != MISS) <= 1.0


@pytest.mark.parametrize("scene", ["one", "instances"])
def test_axis_parallel_rays_on_faces(scenes, scene):
    rng = np.random.default_rng(3)
    n = 20_000
    origin = _edge_points(rng, n)
    off = rng.random(n) < 0.3  # and rays inside the cells
    origin[off, 0:2] = 1.0 + rng.random((int(off.sum()), 2))
    origin[:, 2] = 0.0
    d = np.zeros((n, 3), np.float32)
    d[:, 2] = 1.0
    d[:, 0:2] = np.where(rng.random((n, 2)) < 0.5, np.float32(0.0), np.float32(-0.0))
    pairs = _check(scenes[scene], _rays(origin, d), f"axis {scene}")
    assert 0.2 < np.mean(pairs[:, 0] != MISS) < 1.0


def test_directions_with_large_reciprocals(scenes):
    """Lengths of 2e-19 to 8e-19: 1 / dir is finite and above 2^60."""
    rng = np.random.default_rng(8)
    n = 20_000
    origin = rng.uniform(-3, 3, (n, 3))
    d = np.concatenate([rng.uniform(-1.0, 3.0, (n, 2)), np.full((n, 1), 5.0)], axis=1) - origin
    d *= rng.uniform(2e-19, 8e-19, (n, 1)) / np.linalg.norm(d, axis=1, keepdims=True)
    pairs = _check(scenes["instances"], _rays(origin, d), "short directions")
    assert np.mean(pairs[:, 0] != MISS) > 0.3
