"""Stable compaction at the edges of its tiles and launches: one tile or less,
whole and partial tiles, the largest sum without a scan launch and the smallest
with one, all and nothing kept, the output written over the mask."""

import numpy as np
import pytest

from rendiation_amd.acceleration import AccelerationStructureSystem

pytestmark = pytest.mark.gpu

TILE, DIRECT = 4096, 2048  # elements per tile, tiles without a scan launch


@pytest.mark.parametrize("n", [1, 63, 64, 65, TILE - 1, TILE, TILE + 1, 3 * TILE, 100_003, DIRECT * TILE,
                               DIRECT * TILE + 1])
@pytest.mark.parametrize("density", [0.0, 0.003, 0.4, 1.0])
def test_compaction_is_a_stable_copy_if(device, n, density):
    import torch

    mask = (np.random.default_rng(n).random(n) < density).astype(np.int32) * np.int32(-5)
    want = np.flatnonzero(mask)
    s = AccelerationStructureSystem(device=0)
    for over in (False, True):
        m = torch.from_numpy(mask.copy()).to(device)
        out = m if over else torch.full((n,), -1, dtype=torch.int32, device=device)
        cnt = torch.full((1,), -1, dtype=torch.int32, device=device)
        torch.cuda.synchronize()
        s.compact(m, out, cnt)
        s.sync()
        assert int(cnt.item()) == len(want)
        got = out.cpu().numpy()
        assert np.array_equal(got[:len(want)], want)
        assert over or np.all(got[len(want):] == -1)
    s.close()
