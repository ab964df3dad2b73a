"""Drop-in kernels that take points and cells in runs, at the edges of the
runs: grids of one point or one row per axis, runs that span rows and planes,
arrays that are not 16-byte aligned, and cell counts that end inside a tile."""
import ctypes as C

import numpy as np
import pytest
import torch

from helpers import to_np, ulp_diff
from test_gpu_dropin import compare_with_oracle, grid_args, run_dropin, DropinBuffers

pytestmark = pytest.mark.gpu

POINTS = [(1, 1, 1), (1, 5, 9), (3, 1, 400), (2, 2, 2), (257, 3, 3), (1023, 2, 3), (5, 7, 300),
          (1, 1, 4097), (2049, 1, 1), (2, 1025, 5), (64, 64, 3)]


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("n", POINTS, ids=lambda n: "x".join(map(str, n)))
def test_normalise_four_runs(gc, orc, dev, n, shift):
    npts = n[0] * n[1] * n[2]
    vol = np.random.default_rng(npts).standard_normal(npts).astype(np.float32)
    bufs = [torch.full((npts + 8,), -9.0, dtype=torch.float32, device=dev) for _ in range(3)]
    f, ind, nrm = (b[shift:shift + npts] for b in bufs)
    f.copy_(torch.from_numpy(vol))
    gc.check(gc.lib.gpucad_normalise_four(gc.ptr(f), gc.ptr(ind), gc.ptr(nrm), npts, *n, 0.2, 0.6))
    r_ind, r_nrm = orc.normalise_four(vol, *n, 0.2, 0.6)
    assert np.array_equal(to_np(ind).view(np.uint32), r_ind.view(np.uint32))
    assert np.array_equal(to_np(nrm).view(np.uint32), r_nrm.view(np.uint32))
    for b in bufs:
        assert (b[:shift] == -9).all() and (b[shift + npts:] == -9).all()


@pytest.mark.parametrize("n", POINTS, ids=lambda n: "x".join(map(str, n)))
def test_primitive_runs(gc, orc, dev, n):
    npts = n[0] * n[1] * n[2]
    d, c, a, w = (0.05, 0.06, 0.07), (0.1, -0.05, 0.02), (0.3, -0.2, 0.5), [0.7, 0.5, 0.9]
    out = torch.full((npts + 8,), -9.0, dtype=torch.float32, device=dev)
    gc.check(gc.lib.gpucad_cuboid(gc.ptr(out), gc.Float3(*c), gc.Float3(*a), *w, *n, *d))
    ref = orc.primitive(1, *n, d, c, a, w, 0)
    # within one ulp, the bound of the primitives' test on one shape
    assert ulp_diff(to_np(out)[:npts], ref).max() <= 1
    assert (out[npts:] == -9).all()


CELLS = [(2, 2, 5000), (34, 3, 100), (66, 9, 50), (3, 3, 3), (2, 2, 2), (4098, 2, 3), (33, 2, 300),
         (32, 33, 34), (65, 65, 5)]


@pytest.mark.parametrize("n", CELLS, ids=lambda n: "x".join(map(str, n)))
def test_tile_sums_runs(gc, orc, dev, n):
    npts = n[0] * n[1] * n[2]
    vol = np.random.default_rng(npts + 1).standard_normal(npts).astype(np.float32)
    f = torch.from_numpy(vol).to(dev)
    ref = orc.compute_isosurface(2, vol, *n, 0.1)
    b, active, total = run_dropin(gc, "standard", f, *n, 0.1, max_verts=max(npts * 16, 300000))
    compare_with_oracle(orc, b, active, total, ref, check_pos=False)
    # the first cells only: the last tile ends inside a row
    cells = (n[0] - 1) * (n[1] - 1) * (n[2] - 1)
    part = max(1, cells - 37)
    b = DropinBuffers(cells, 300000, dev)
    active, total = C.c_uint32(0), C.c_uint32(0)
    gs, sh, mk = grid_args(gc, *n)
    one = gc.Float3(1, 1, 1)
    gc.check(gc.lib.gpucad_compute_isosurface_standard(
        gc.ptr(f), gc.ptr(b.pos), gc.ptr(b.norm), 0.1, part, gc.ptr(b.verts),
        gc.ptr(b.verts_scan), gc.ptr(b.occ), gc.ptr(b.occ_scan), gs, sh, mk, one, one,
        C.byref(active), C.byref(total), gc.ptr(b.comp), 300000))
    v = ref["verts"][:part].astype(np.int64)
    assert (active.value, total.value) == (int((v > 0).sum()), int(v.sum()))
    assert np.array_equal(to_np(b.verts)[:part].astype(np.int64), v)
    scan = np.concatenate([[0], np.cumsum(v)[:-1]])
    if active.value:
        assert np.array_equal(to_np(b.verts_scan)[:part].astype(np.int64), scan)
