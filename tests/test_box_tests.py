"""The box tests of the traversal (csrc/box_test.h, compiled here for the host):
the form that the child-quad layouts use, near and far planes chosen by the
direction's sign, gives the reference's slab test, also at box edges and for
origins small against the planes, where another rounding would decide
otherwise; the decoded planes of a quantized node are corner + q * step."""

import ctypes
import subprocess

import numpy as np
import pytest

from tests.conftest import ROOT

SOURCE = r"""
#include "box_test.h"
using namespace rdrt;
extern "C" void tests(long n, const float *ray, const float *box, float *tn, unsigned char *out) {
  for (long i = 0; i < n; i++) {
    const float *r = ray + 8 * i, *b = box + 6 * i;
    const F3 o{r[0], r[1], r[2]}, inv{1.0f / r[4], 1.0f / r[5], 1.0f / r[6]};
    out[3 * i] = slab(o, inv, r[3], r[7], b[0], b[1], b[2], b[3], b[4], b[5], tn[2 * i]);
    const RayBox q = ray_box(o, inv);
    const bool sx = std::signbit(inv.x), sy = std::signbit(inv.y), sz = std::signbit(inv.z);
    const float nx = b[sx ? 3 : 0], fx = b[sx ? 0 : 3], ny = b[sy ? 4 : 1], fy = b[sy ? 1 : 4], nz = b[sz ? 5 : 2],
                fz = b[sz ? 2 : 5];
    out[3 * i + 1] = q.plain ? planes_hit<true>(q, r[3], r[7], nx, ny, nz, fx, fy, fz, tn[2 * i + 1])
                             : planes_hit<false>(q, r[3], r[7], nx, ny, nz, fx, fy, fz, tn[2 * i + 1]);
    out[3 * i + 2] = q.plain;
  }
}
extern "C" void decode(long n, const float *corner, const float *step, const unsigned *word, float *out) {
  for (long i = 0; i < n; i++)
    for (int c = 0; c < 4; c++) {
      const float v = (float)((word[i] >> (8 * c)) & 0xffu) * step[i];
      out[8 * i + c] = corner[i] + v;
      out[8 * i + 4 + c] = dequant(corner[i], word[i], c, step[i]);
    }
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("box")
    (d / "box.cpp").write_text("#include <cmath>\n" + SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared", "-Wall", "-Werror",
                    f"-I{ROOT / 'rendiation_amd' / 'csrc'}", str(d / "box.cpp"), "-o", str(d / "box.so")], check=True)
    return ctypes.CDLL(str(d / "box.so"))


def _run(lib, ray, box):
    n = len(ray)
    ray, box = np.ascontiguousarray(ray, np.float32), np.ascontiguousarray(box, np.float32)
    tn, out = np.empty((n, 2), np.float32), np.empty((n, 3), np.uint8)
    lib.tests(ctypes.c_long(n), *(a.ctypes.data_as(ctypes.c_void_p) for a in (ray, box, tn, out)))
    return tn, out.astype(bool)


def _same(lib, ray, box):
    tn, out = _run(lib, ray, box)
    assert np.array_equal(out[:, 0], out[:, 1])
    hit = out[:, 0]
    assert np.array_equal(tn[hit, 0], tn[hit, 1])
    return out


def _boxes(rng, n):
    a, b = rng.uniform(-2, 2, (n, 3)), rng.uniform(-2, 2, (n, 3))
    grid = rng.random(n) < 0.5
    a[grid], b[grid] = np.round(a[grid] * 8) / 8, np.round(b[grid] * 8) / 8
    flat = rng.random((n, 3)) < 0.2
    b = np.where(flat, a, b)
    return np.concatenate([np.minimum(a, b), np.maximum(a, b)], axis=1).astype(np.float32)


@pytest.mark.parametrize("size", [0.0, 1e-6, 1e-3, 0.05, 0.25, 1.0, 10.0])
def test_rays_aimed_at_box_edges(lib, size):
    rng = np.random.default_rng(int(size * 1e6) + 1)
    n = 400_000
    box = _boxes(rng, n)
    ray = np.zeros((n, 8), np.float32)
    ray[:, 0:3] = rng.uniform(-1, 1, (n, 3)) * size
    at = box.reshape(n, 2, 3)[np.arange(n)[:, None], rng.integers(0, 2, (n, 3)), np.arange(3)]  # a corner
    inner = rng.random((n, 3)) < 0.4  # or a point of an edge, a face, the inside
    at = np.where(inner, box[:, :3] + rng.random((n, 3)) * (box[:, 3:] - box[:, :3]), at).astype(np.float32)
    ray[:, 4:7] = at - ray[:, 0:3]
    ray[:, 7] = np.inf
    out = _same(lib, ray, box)
    assert 0.2 < out[:, 0].mean() < 0.999
    assert size == 0.0 or out[:, 2].mean() > 0.5


def test_axis_parallel_tiny_and_extreme_rays(lib):
    rng = np.random.default_rng(5)
    n = 400_000
    box = _boxes(rng, n)
    ray = np.zeros((n, 8), np.float32)
    ray[:, 0:3] = rng.uniform(-2.5, 2.5, (n, 3))
    on = rng.random((n, 3)) < 0.3  # the origin on a face's plane: 0 * inf where the direction is parallel to it
    ray[:, 0:3] = np.where(on, box[:, :3], ray[:, 0:3])
    special = np.array([0.0, -0.0, 1e-19, -1e-30, 1e-42, np.inf, -np.inf, np.nan, 1e30], np.float32)
    d = rng.uniform(-1, 1, (n, 3)).astype(np.float32)
    d = np.where(rng.random((n, 3)) < 0.6, special[rng.integers(0, len(special), (n, 3))], d)
    d[: n // 2] = np.where(np.abs(d[: n // 2]) > 1.0, np.float32(0.0), d[: n // 2])
    ray[:, 4:7] = d
    ray[:, 3], ray[:, 7] = rng.choice([0.0, 1e-4, -1.0], n), rng.choice([np.inf, 3.0], n)
    out = _same(lib, ray, box)
    assert 1000 < out[:, 0].sum() and out[:, 2].any() and not out[:, 2].all()


def test_decoded_planes(lib):
    rng = np.random.default_rng(9)
    n = 200_000
    corner = (rng.uniform(-1, 1, n) * 10.0 ** rng.integers(-6, 7, n)).astype(np.float32)
    step = np.ldexp(np.float32(1.0), rng.integers(-126, 100, n)).astype(np.float32)
    step[:100] = np.finfo(np.float32).max  # the step of an axis that no power of two fits
    word = rng.integers(0, 2**32, n, dtype=np.uint32)
    out = np.empty((n, 8), np.float32)
    lib.decode(ctypes.c_long(n), *(a.ctypes.data_as(ctypes.c_void_p) for a in (corner, step, word, out)))
    assert np.array_equal(out[:, :4], out[:, 4:])
