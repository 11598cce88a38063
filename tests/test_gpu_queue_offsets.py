"""Queues compacted without a scan launch: the rays that a cull pass keeps, at
the edges of a block and of the most blocks that sum their offsets themselves,
with no ray, some rays and every ray kept."""

import numpy as np
import pytest

from rendiation_amd import synth
from rendiation_amd.acceleration import (AccelerationStructureSystem, TopLevelAccelerationStructureSourceInstance,
                                         TriangleGeometry)

pytestmark = pytest.mark.gpu

BLOCK, DIRECT = 256, 4096  # rays per block, blocks without a scan launch


@pytest.mark.parametrize("n", [1, BLOCK, BLOCK + 1, 100_003, DIRECT * BLOCK, DIRECT * BLOCK + 1])
def test_culled_trace_equals_plain(device, n):
    import torch

    s = AccelerationStructureSystem(device=0)
    b = s.create_bottom_level_acceleration_structure([TriangleGeometry(synth.random_triangles(0, 500, spread=0.3))])
    s.bind_tlas([s.create_top_level_acceleration_structure(
        [TopLevelAccelerationStructureSourceInstance(np.eye(4), b)])])
    s.build()
    s.create_comp_instance()
    away = np.zeros((n, 8), np.float32)
    away[:, 0], away[:, 3], away[:, 4], away[:, 7] = 50.0, 1e-4, 1.0, np.inf  # from outside, outwards
    some = away.copy()
    some[::3] = synth.random_rays(1, n)[::3]
    for name, rays_np in (("none", away), ("some", some), ("all", synth.random_rays(2, n))):
        print(f"[gpu-case] cull pass, {n} rays, {name} kept", flush=True)
        rays = torch.from_numpy(rays_np).to(device)
        got = []
        for cull in (0, 1):
            s.set_tune(cull=cull)
            hits = torch.full((n, 4), 7, dtype=torch.int32, device=device)
            torch.cuda.synchronize()
            s.trace(rays, hits)
            s.sync()
            got.append(hits.cpu().numpy())
        assert np.array_equal(got[0], got[1]), name
    s.close()
