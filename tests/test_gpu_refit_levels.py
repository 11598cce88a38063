"""Refit at the edges of its level launches: one triangle, chains of more
levels than one launch takes, levels about the width of a block, and repeated
refits (the second writes the TLAS layer in place)."""

import numpy as np
import pytest

from rendiation_amd import synth
from rendiation_amd.acceleration import TRAVERSAL_REFERENCE
from tests.parity import compare
from tests.test_gpu_wave_traversal import _ladder, _system, _trace

pytestmark = pytest.mark.gpu


def _scene(kind):
    if kind == "ladder":
        return _ladder(40)
    n = {"one": 1, "block": 1030, "wide": 5000}[kind]
    return synth.random_triangles(21, n, spread=0.05)


@pytest.mark.parametrize("kind", ["one", "ladder", "block", "wide"])
def test_refit_levels(device, kind):
    import torch

    pos = _scene(kind)
    m = np.eye(4)
    m[:3, 3] = [0.3, 0.1, -0.2]
    s = _system([(pos, None)], [np.eye(4), m], blas_bin_size=1)
    scale = np.float32(1000.0 if kind == "ladder" else 1.0)
    rays = synth.random_rays(6, 6000, lo=-0.3, hi=1.6)
    rays[:, 0:3] *= scale
    for step in range(3):  # away, elsewhere, back
        moved = pos if step == 2 else (pos * np.float32(1.0 + 0.3 * (step + 1)) + np.float32(0.05)).astype(np.float32)
        print(f"[gpu-case] refit {kind} step {step}", flush=True)
        s.refit(torch.from_numpy(moved).cuda())
        fresh = _system([(moved, None)], [np.eye(4), m], blas_bin_size=1)
        want = _trace(fresh, rays, TRAVERSAL_REFERENCE)
        for shape in ((256, 16, 0, 0, 0, 0), (64, 8, 6, 1, 0, 1), (128, 16, 6, 0, 0, 2)):
            s.set_tune(*shape)
            d = compare(_trace(s, rays, 0), want)
            assert d.ok() and d.value_mismatch_bits == 0, (kind, step, shape, d)
        assert compare(_trace(s, rays, TRAVERSAL_REFERENCE), want).ok()
        fresh.close()
    s.close()
