"""The traversal's per-lane stack: one inner step from every fill level, lanes
alone and together, against a list.  Entries past its end are dropped and
raise the status bit, in every variant."""

import ctypes
from pathlib import Path

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIB = Path(__file__).resolve().parent / "stages" / "libstack_stages.so"
WORDS = 64


def _step(lds, entries, layout, sp, kids):
    import torch

    lib = ctypes.CDLL(str(LIB))
    a = [torch.from_numpy(np.asarray(v, dtype=np.int32)).cuda() for v in (sp, kids)]
    status = torch.zeros(64, dtype=torch.int32, device="cuda")
    out = torch.full((64, WORDS), -1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    rc = lib.stack_step(ctypes.c_uint32(lds), ctypes.c_uint32(entries), ctypes.c_uint32(layout),
                        *(ctypes.c_void_p(t.data_ptr()) for t in (*a, status, out)), ctypes.c_uint32(WORDS))
    assert rc == 0
    torch.cuda.synchronize()
    return status.cpu().numpy(), out.cpu().numpy()


def _expect(limit, sp, n):
    stack = [100 + i for i in range(sp)]
    if n == 0:
        return stack[:-1], stack[-1], 0
    stack += list(range(1, n))
    return stack[:limit], n, int(len(stack) > limit)


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("lds,entries", [(8, 8), (16, 16), (8, 24), (16, 48)])
def test_step_from_every_level(device, lds, entries, layout):
    limit, most = entries + 2, 2 if layout == 0 else 4  # two end marks beside the refs
    cases = [(sp, n) for sp in range(1, limit + 1) for n in range(most + 1)]
    mixed = np.random.default_rng(entries).permutation(len(cases))
    waves = [[c] * 64 for c in cases] + [[cases[mixed[(k + i) % len(cases)]] for i in range(64)]
                                        for k in range(0, len(cases), 64)]
    for wave in waves:
        status, out = _step(lds, entries, layout, [c[0] for c in wave], [c[1] for c in wave])
        for lane, (sp, n) in enumerate(wave):
            stack, ref, over = _expect(limit, sp, n)
            assert (out[lane, 0], out[lane, 1], status[lane]) == (len(stack), ref, over), (sp, n)
            assert out[lane, 2:2 + len(stack)].tolist() == stack, (sp, n)
