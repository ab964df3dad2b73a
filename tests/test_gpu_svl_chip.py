"""The phase solve that keeps its vectors on the chip (one launch, tiles split
along y and z), the unit cell's separable spectrum and the fused synthesis at
the sizes where they can go wrong: the smallest grids, tiles of two rows or
planes, runs of every length modulo four, one tile, several right-hand sides,
grids too wide for a tile (the two-launch form), every coefficient range,
ragged fine rows.

Tolerances: the solve's own, as in test_gpu_svl (the iterations are the
oracle's within 5 %, the solution within 2 % of its largest value); the
spectrum's FP64 sums round once to FP32 (1e-6 of the largest coefficient); the
synthesis against the oracle's from the same solves, within what their
residuals allow (2 % of the largest value, 0.2 % on average)."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DIMS = [(4, 4, 4), (5, 4, 6), (7, 5, 23), (12, 33, 9), (33, 37, 50), (128, 17, 9), (61, 57, 70),
        (120, 24, 25), (255, 9, 11), (512, 4, 6), (520, 5, 4)]


@pytest.mark.parametrize("dims", DIMS)
def test_cg_tiles_against_oracle(gc, orc, dev, dims):
    b = orc.svl_finding_phi(*dims, 1, -2, 1, lattice_type="b", uniform_type=0, const_period=9.0)
    xo, ito, _ = orc.svl_cg(b, *dims, iters=400, end_res=0.02)
    d = torch.from_numpy(b.copy()).to(dev)
    it, res = C.c_int32(0), C.c_float(0)
    for _ in range(2):  # (the second solve finds the first one's exchange words)
        d.copy_(torch.from_numpy(b))
        gc.check(gc.lib.gpucad_svl_cg(gc.ptr(d), *dims, 400, 0.02, C.byref(it), C.byref(res)))
        x = d.cpu().numpy()
        assert abs(it.value - ito) <= max(2, ito // 20)
        assert it.value == 400 or res.value <= 0.02
        assert np.max(np.abs(x - xo)) < 2e-2 * np.max(np.abs(xo))


@pytest.mark.parametrize("dims", [(4, 4, 4), (30, 21, 18), (40, 96, 44)])
def test_three_right_hand_sides_stop_alone(gc, orc, dev, dims):
    """One solve of three right-hand sides against three of one each."""
    nx, ny, nz = dims
    p = gc.svl_params(nx, lattice_type="r", const_period=11.0, range_=1, cg_end_res=0.03)
    p.ny, p.nz, p.fy, p.fz = ny, nz, 2 * ny, 2 * nz
    _, got = gc.svl_field(p, torch.zeros(27, dtype=torch.complex64, device=dev))
    tol = np.float32(0.03) / np.float32(3)
    for a, ijk in enumerate(((1, 0, 0), (0, 1, 0), (0, 0, 1))):
        b = orc.svl_finding_phi(*dims, *ijk, lattice_type="r", uniform_type=0, const_period=11.0)
        d = torch.from_numpy(b).to(dev)
        it, res = C.c_int32(0), C.c_float(0)
        gc.check(gc.lib.gpucad_svl_cg(gc.ptr(d), *dims, 500, tol, C.byref(it), C.byref(res)))
        assert abs(got.cg_iters[a] - it.value) <= 1
        assert got.cg_res[a] <= tol


@pytest.mark.parametrize("dims,r", [((61, 61, 61), 2), ((5, 7, 3), 4), ((130, 3, 2), 3),
                                    ((1, 1, 1), 0), ((64, 65, 9), 1), ((3, 70, 67), 4)])
def test_unit_spectrum_shapes(gc, orc, dev, dims, r):
    nx, ny, nz = dims
    cell = np.random.default_rng(21).standard_normal(nx * ny * nz).astype(np.float32)
    out = torch.zeros((2 * r + 1) ** 3, dtype=torch.complex64, device=dev)
    gc.check(gc.lib.gpucad_unit_spectrum(gc.ptr(torch.from_numpy(cell).to(dev)), nx, ny, nz, r,
                                         gc.ptr(out)))
    ref = orc.unit_spectrum(cell, nx, ny, nz, r)
    assert np.max(np.abs(out.cpu().numpy() - ref)) < 1e-6 * max(1.0, np.max(np.abs(ref)))


@pytest.mark.parametrize("n,r,harmonics,fx", [(9, 0, 1, 18), (8, 1, 27, 15), (10, 2, 62, 20),
                                              (7, 3, 200, 13), (6, 4, 729, 12), (136, 2, 62, 270)])
def test_synthesis_ranges(gc, orc, dev, n, r, harmonics, fx):
    p = gc.svl_params(n, lattice_type="b", const_period=7.0, range_=r, harmonics=harmonics,
                      cg_end_res=1e-3, cg_max_iter=3000)
    p.ny, p.nz, p.fx, p.fy, p.fz = 6, 5, fx, 11, 9
    c = np.random.default_rng(22).standard_normal(((2 * r + 1) ** 3, 2)).astype(np.float32)
    svl, res = gc.svl_field(p, torch.from_numpy(c).to(dev))
    ref, _, _ = orc.svl_field(p, c, None)
    scale = max(1e-3, np.max(np.abs(ref)))
    out = svl.cpu().numpy()
    assert np.max(np.abs(out - ref)) < 2e-2 * scale
    assert np.mean(np.abs(out - ref)) < 2e-3 * scale
