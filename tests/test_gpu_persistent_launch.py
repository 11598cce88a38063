"""Persistent traversal launches: an empty one ends at once, and every ray is
traced once where the XCDs' shares of the queue are uneven, empty or smaller
than the first chunks of their waves."""

import numpy as np
import pytest

from rendiation_amd import synth
from rendiation_amd.acceleration import TRAVERSAL_FAST, TRAVERSAL_REFERENCE
from tests.parity import MISS, compare
from tests.test_gpu_wave_traversal import _say, _system, _trace

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def system(device):
    s = _system([(synth.random_triangles(3, 2000, spread=0.05), None)], blas_bin_size=4)
    yield s
    s.close()


def test_empty_launch_costs_as_much_as_a_plain_one(system):
    """The cull pass finishes every ray, so the traversal launch finds none.
    Its waves must not queue up on the work counters: a thousand waves that
    add to one address take some 18 us, the whole empty launch about 5."""
    import torch

    n = 400_000
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0], rays[:, 3], rays[:, 4], rays[:, 7] = 50.0, 1e-4, 1.0, np.inf  # outwards, from outside
    r = torch.from_numpy(rays).cuda()
    hits = torch.empty((n, 4), dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    best = {}
    for _ in range(7):
        for persist in (0, 1):
            system.set_tune(64, 16, 6, persist, 1, 1)
            e0, e1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            for k in range(60):
                if k == 10:
                    e0.record()
                system.trace(r, hits)
            e1.record()
            system.sync()
            torch.cuda.synchronize()
            us = e0.elapsed_time(e1) * 1e3 / 50
            best[persist] = min(us, best.get(persist, us))
    _say(f"empty launch: plain {best[0]:.1f} us, persistent {best[1]:.1f} us")
    assert bool((hits[:, 0] == -1).all())  # MISS
    # both sides hold the cull pass; the clearing launch of the counters comes on top of a persistent one
    assert best[1] <= best[0] + 15.0, best


@pytest.mark.parametrize("block", [64, 256])
def test_uneven_shares(system, block):
    rng = np.random.default_rng(block)
    for n in [1, 7, 8, 9, 64, 511, 512, 513, 520, 4095, 4097, 33_000, 131_071, 700_001]:
        rays = synth.random_rays(n, n, lo=-0.2, hi=1.2)
        want = _trace(system, rays, TRAVERSAL_REFERENCE)
        for wide, cull in ((0, 0), (1, 0), (1, 1), (2, 1)):
            _say(f"persistent block {block} wide {wide} cull {cull} n={n}")
            system.set_tune(block, int(rng.choice([8, 16])), int(rng.choice([0, 6])), 1, cull, wide)
            d = compare(_trace(system, rays, TRAVERSAL_FAST), want)
            assert d.ok() and d.value_mismatch_bits == 0, (n, wide, d)
    assert np.count_nonzero(want[:, 0] != MISS) > 1000
