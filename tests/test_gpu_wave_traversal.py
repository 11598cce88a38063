"""The one-ray-per-lane traversal kernels against the reference-order kernel
(itself bit-exact with the oracle) where their wave scheduling, stack and node
tests can go wrong: partial waves and refills, stacks deeper than their LDS
rows, axis-parallel rays, leaves of several instances, several geometries."""

import numpy as np
import pytest

from rendiation_amd import synth
from rendiation_amd.acceleration import (
    RAY_FLAG_ACCEPT_FIRST_HIT_AND_END_SEARCH,
    TRAVERSAL_FAST,
    TRAVERSAL_REFERENCE,
    AccelerationStructureSystem,
    BuildOptions,
    TopLevelAccelerationStructureSourceInstance,
    TriangleGeometry,
)
from tests.parity import MISS, compare

pytestmark = pytest.mark.gpu

SHAPES = [(b, lds, w, p, 0, wide, coop) for wide in (0, 1, 2)
          for b, lds, w, p, coop in ((64, 8, 0, 0, 0), (256, 16, 6, 1, 0), (128, 8, 6, 1, 0), (64, 8, 6, 0, 1 << 20))]


def _say(msg):
    print(f"[gpu-case] {msg}", flush=True)


def _system(geometries, transforms=(np.eye(4),), **options):
    s = AccelerationStructureSystem(device=0, options=BuildOptions(**options))
    b = s.create_bottom_level_acceleration_structure([TriangleGeometry(p, i) for p, i in geometries])
    t = s.create_top_level_acceleration_structure(
        [TopLevelAccelerationStructureSourceInstance(m, b) for m in transforms])
    s.bind_tlas([t])
    s.create_comp_instance()
    return s


def _trace(s, rays, traversal, **kw):
    import torch

    r = torch.from_numpy(rays).to("cuda:0")
    hits = torch.full((len(rays), 4), -7, dtype=torch.int32, device="cuda:0")
    torch.cuda.synchronize()
    s.trace(r, hits, traversal=traversal, **kw)
    s.sync()
    return hits.cpu().numpy().view(np.uint32)


def _check(s, rays, what):
    want = _trace(s, rays, TRAVERSAL_REFERENCE)
    for shape in SHAPES:
        _say(f"{what} {shape} n={len(rays)}")
        s.set_tune(*shape)
        d = compare(_trace(s, rays, TRAVERSAL_FAST), want)
        assert d.ok() and d.value_mismatch_bits == 0, (what, shape, d)
        any_hit = _trace(s, rays, TRAVERSAL_FAST, flags=RAY_FLAG_ACCEPT_FIRST_HIT_AND_END_SEARCH)
        assert np.array_equal(any_hit[:, 0] == MISS, want[:, 0] == MISS), (what, shape)
    return want


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000, 4097, 70_001])
def test_ray_counts(device, n):
    s = _system([(synth.random_triangles(3, 3000, spread=0.03), None)], blas_bin_size=4)
    want = _check(s, synth.random_rays(5, n, lo=-0.2, hi=1.2), "counts")
    assert n < 1000 or 0 < np.count_nonzero(want[:, 0] != MISS) < n
    s.close()


def _ladder(count):
    """Triangles across the x axis at x = 2^(10 - i), sized by x: the trees are chains, whose quads need stacks of 16,
    24 and 48 entries for 12, 24 and 40 triangles.  (The products of four edge lengths stay normal numbers.)"""
    x = np.float32(2.0) ** (10 - np.arange(count, dtype=np.float32))
    tri = np.zeros((count, 3, 3), dtype=np.float32)
    tri[:, :, 0] = x[:, None]
    tri[:, :, 1:] = np.array([[-1.0, -1.0], [1.0, -1.0], [0.0, 1.2]], dtype=np.float32) * x[:, None, None]
    return tri.reshape(-1, 3)


@pytest.mark.parametrize("count,entries", [(12, 16), (24, 24), (40, 48)])
def test_deep_stacks(device, count, entries):
    s = _system([(_ladder(count), None)], blas_bin_size=1)
    assert s.scene_info().quad_stack_entries == entries
    rng = np.random.default_rng(count)
    n = 4096
    size = np.float32(2.0) ** (10 - rng.uniform(0.0, count, n))
    rays = np.zeros((n, 8), dtype=np.float32)
    rays[:, 0] = np.where(rng.random(n) < 0.7, -1.0, 2000.0)  # towards the small end: the deepest child is the nearest
    rays[:, 1:3] = rng.uniform(-1.2, 1.2, (n, 2)) * size[:, None]
    rays[:, 4] = np.where(rays[:, 0] < 0, 1.0, -1.0)
    rays[:, 5:7] = rng.uniform(-1e-4, 1e-4, (n, 2)) * size[:, None]
    rays[:, 3], rays[:, 7] = 1e-6, np.inf
    want = _check(s, rays, "ladder")
    assert len(np.unique(want[:, 0])) > count // 2
    s.close()


def test_axis_parallel_rays(device):
    pos, idx, _ = synth.height_field(40, seed=2, amplitude=0.1)
    s = _system([(pos, idx)], [np.eye(4), np.diag([2.0, 1.0, 2.0, 1.0])])
    rng = np.random.default_rng(1)
    n = 3000
    rays = np.zeros((n, 8), dtype=np.float32)
    rays[:, 0:3] = rng.uniform(-1.9, 1.9, (n, 3))
    axis = rng.integers(0, 3, n)
    rays[np.arange(n), 4 + axis] = np.where(rng.random(n) < 0.5, 1.0, -1.0)
    neg = rng.random((n, 3)) < 0.5  # zeros of both signs
    rays[:, 4:7] = np.where((rays[:, 4:7] == 0.0) & neg, np.float32(-0.0), rays[:, 4:7])
    rays[: n // 3, 4] += np.float32(1e-20)  # and tiny components, whose reciprocals are huge
    rays[:, 3], rays[:, 7] = 1e-4, 100.0
    want = _check(s, rays, "axis-parallel")
    assert np.count_nonzero(want[:, 0] != MISS) > 100
    s.close()


def test_leaves_of_several_instances_and_geometries(device):
    sph_p, sph_i = synth.uv_sphere(20, 10)
    tor_p, tor_i = synth.torus(24, 8)
    rng = np.random.default_rng(4)
    ts = []
    for k in range(11):
        m = np.eye(4)
        m[:3, :3] = synth.random_rotation(7, 1, k) * rng.uniform(0.5, 1.5)
        m[:3, 3] = rng.uniform(-2, 2, 3)
        ts.append(m)
    # a TLAS depth bound leaves several instances in one leaf
    s = _system([(sph_p * np.float32(0.5), sph_i), (tor_p, tor_i), (sph_p * np.float32(0.1), sph_i)], ts,
                tlas_max_depth=1, tlas_bin_size=1)
    _check(s, synth.random_rays(9, 20_000, lo=-3.0, hi=3.0), "instances")
    s.close()
