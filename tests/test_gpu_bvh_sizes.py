"""The device's binned-SAH hierarchy against the oracle's, word for word, at
the sizes where the builder changes its way of working: one 16-lane group, one
wave, one chunk and several levels of chunks; with triangles that no axis
separates (halved in index order)."""
import ctypes as C

import numpy as np
import pytest

import orc
from risltc_amd import synth

pytestmark = pytest.mark.gpu


def triangles(n, kind, rng):
    small = rng.normal(0, 0.3, (n, 3, 3))
    if kind == "same":
        return np.broadcast_to(small[:1], (n, 3, 3)).copy()  # one place, n times
    centre = rng.uniform(-20, 20, (n, 1, 3))
    if kind == "line":
        centre[:, :, 1:] = 1.0
        small[:, :, 1:] = small[:1, :, 1:]  # two axes without extent
    if kind == "clumps":
        centre = rng.integers(0, 3, (n, 1, 3)) * 5.0 + (rng.random((n, 1, 3)) < 0.3) * 1e-4
        small = np.broadcast_to(small[:1], (n, 3, 3))
    return centre + small


@pytest.mark.parametrize("n", [1, 2, 3, 15, 16, 17, 63, 64, 65, 255, 256, 257, 700, 2047, 2049, 5000, 20011])
@pytest.mark.parametrize("kind", ["spread", "same", "line", "clumps"])
def test_records_equal_the_oracle(n, kind):
    import risltc_amd
    rng = np.random.default_rng(n)
    mesh = synth.Mesh(triangles(n, kind, rng), np.tile(np.array([0.0, 0.0, 1.0]), (n, 3, 1)), np.zeros((n, 3, 2)),
                      np.zeros(n, int), rng.integers(0, 2, n))
    ctx = risltc_amd.Context(0)
    ctx.set_scene(mesh, [[0.5] * 6])
    got = ctx.bvh_records()
    L, bvh = orc.lib(), orc.OrcBvh()
    tri = np.ascontiguousarray(mesh.dequantized(), np.float32)
    L.orc_bvh_build_sah(C.byref(bvh), orc.ptr(tri, orc.f32p), n)
    want = np.zeros((5 * n - 2, 4), np.float32)
    pos = np.ascontiguousarray(mesh.positions, np.uint32)
    L.orc_bvh_records(C.byref(bvh), orc.ptr(pos, orc.u32p), orc.ptr(want, orc.f32p))
    L.orc_bvh_free(C.byref(bvh))
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
