"""Vertex gradient sums at the sizes where their wave-wise scatter can go
wrong: frames of less than a wave, partial waves and blocks, one view and
several, terms with and without normals, against the FP64 oracle."""

import dataclasses

import numpy as np
import pytest

from rendiation_amd.pathtracer import Camera
from rendiation_amd import synth
from tests.pt_util import oracle_params, oracle_scene_from
from tests.test_gpu_grad import GRAD_REL, _rel, geo_case  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height,spp,views,bounces", [(1, 1, 1, 1, 1), (9, 7, 1, 1, 2), (8, 8, 1, 1, 3),
                                                             (65, 3, 1, 1, 2), (16, 16, 3, 3, 1), (31, 33, 2, 1, 3)])
def test_vertex_gradients_of_odd_frames(geo_case, width, height, spp, views, bounces):  # noqa: F811
    import torch

    scene, system, tracer, _, cfg, _ = geo_case
    print(f"[gpu-case] {width}x{height} spp {spp} views {views} bounces {bounces}", flush=True)
    cams = [Camera(position=p, aspect=1.0) for p in synth.sphere_views(3, radius=2.5)][:views]
    cfg = dataclasses.replace(cfg, width=width, height=height, spp=spp, max_bounces=bounces, rr_start=bounces)
    adj = np.random.default_rng(width).uniform(0.5, 1.0, size=(views, height, width, 3))
    nv = system.scene_info().verts
    tracer.render(cams, cfg)
    g_pos = torch.full((nv, 3), 7.0, dtype=torch.float32, device="cuda")
    g_nrm = torch.full((nv, 3), 7.0, dtype=torch.float32, device="cuda")
    tracer.backward_geometry(torch.from_numpy(adj.astype(np.float32)).cuda(), g_pos, g_nrm)
    torch.cuda.synchronize()
    op, on = oracle_scene_from(scene).pt_grad_geometry(oracle_params(cams, cfg), adj.reshape(-1, width, 3))
    for got, want in ((g_pos, op), (g_nrm, on)):
        got = got.cpu().numpy().astype(np.float64)
        # an entry without a term is exactly zero, the others agree as sums of 32-bit terms do
        assert np.all(got[want == 0.0] == 0.0)
        assert _rel(got, want) <= GRAD_REL if np.any(want) else not np.any(got)
