"""The phase solve's two forms against each other and the oracle: a solve on the
chip counts as done only when every tile wrote its part, a solve that gives up
is made by two launches from the same right-hand sides, and every kernel of
the chip form with one to three passes over a tile's y halo.

Both forms do the oracle's arithmetic per point, and alpha and beta are sums
in FP64 rounded once, so they differ from the oracle's by one rounding now and
then (6e-8 of a coefficient): over at most 20 iterations the solutions agree
within 1e-4 of the largest value."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

TWO_LAUNCH, ON_CHIP = 1, 2


def solve(gc, dev, b, dims, iters, end_res, form=0, wait_first=0.0, wait=0.0):
    """b: (m, n) right-hand sides; returns x (m, n), iterations, residuals, how."""
    m = len(b)
    d = torch.from_numpy(np.ascontiguousarray(b)).to(dev)
    it, res, how = (C.c_int32 * m)(), (C.c_float * m)(), (C.c_int32 * 5)()
    gc.check(gc.lib.gpucad_svl_cg_form(gc.ptr(d), m, *dims, iters, end_res, form, wait_first, wait,
                                       it, res, how))
    return d.cpu().numpy(), list(it), list(res), list(how)


def rhs(orc, dims, m):
    ijk = ((1, -2, 1), (0, 1, 0), (2, 0, -1), (0, 0, 1))
    return np.stack([orc.svl_finding_phi(*dims, *ijk[a], lattice_type="b", uniform_type=0,
                                         const_period=9.0) for a in range(m)])


@pytest.mark.parametrize("m", [1, 3])
@pytest.mark.parametrize("first", [0.0, -1.0], ids=["first tile waits", "no tile waits"])
def test_a_tile_that_leaves_makes_the_solve_unfinished(gc, orc, dev, m, first):
    dims = (40, 24, 40)
    b = rhs(orc, dims, m)
    zero = np.zeros_like(b)
    for c, iters, end_res in ((zero, 50, 0.01), (b, 1, 0.0), (b, 50, 1e9), (b, 12, 0.0)):
        want = solve(gc, dev, c, dims, iters, end_res, TWO_LAUNCH)
        # (leaves another solution where the next solve keeps its own)
        assert solve(gc, dev, b, dims, 12, 0.0, ON_CHIP)[3][0] == ON_CHIP
        # the other tiles post their sums and leave at their first wait
        got = solve(gc, dev, c, dims, iters, end_res, ON_CHIP, first, -1.0)
        assert got[3][0] == TWO_LAUNCH
        assert np.array_equal(got[0], want[0]) and got[1:3] == want[1:3]
    assert solve(gc, dev, b, dims, 12, 0.0, ON_CHIP)[3][0] == ON_CHIP


# dims, m, planes of a tile rounded up to 4, passes over a y halo
PLANS = [((12, 12, 12), 1, 4, 1), ((61, 57, 70), 1, 8, 1), ((255, 33, 80), 1, 8, 2),
         ((90, 90, 90), 3, 12, 1), ((120, 120, 120), 1, 12, 2), ((128, 128, 128), 2, 16, 2),
         ((119, 101, 93), 3, 16, 2), ((150, 150, 150), 1, 16, 3), ((110, 110, 110), 3, 20, 3),
         ((120, 120, 120), 3, 24, 3), ((33, 37, 50), 4, 4, 1)]


@pytest.mark.parametrize("dims,m,planes,passes", PLANS)
def test_the_forms_agree(gc, orc, dev, dims, m, planes, passes):
    b = rhs(orc, dims, m)
    if m > 1:
        b[-1] *= np.float32(2.0 ** -9)  # stops before the others
    end_res = float(np.linalg.norm(b[-1].astype(np.float64))) * 0.7
    chip = solve(gc, dev, b, dims, 9, end_res, ON_CHIP)
    assert chip[3][0] == ON_CHIP and chip[3][3:] == [planes, passes]
    two = solve(gc, dev, b, dims, 9, end_res, TWO_LAUNCH)
    assert two[3][0] == TWO_LAUNCH
    assert chip[1] == two[1]
    for s in range(m):
        xo, ito, reso = orc.svl_cg(b[s], *dims, iters=9, end_res=end_res)
        for x, it, res, _ in (chip, two):
            assert it[s] == ito
            assert abs(res[s] - reso) <= 1e-4 * reso
            assert np.max(np.abs(x[s] - xo)) <= 1e-4 * np.max(np.abs(xo))


@pytest.mark.parametrize("dims,m", [((520, 40, 30), 3), ((170, 170, 170), 1)])
def test_grids_past_the_chip(gc, orc, dev, dims, m):
    """Rows too wide for a tile, or too many points: several right-hand sides
    and steps per workgroup in the two-launch form."""
    b = rhs(orc, dims, m)
    with pytest.raises(gc.GpucadError):
        solve(gc, dev, b, dims, 9, 0.0, ON_CHIP)
    x, it, res, how = solve(gc, dev, b, dims, 9, 0.0)
    assert how[:3] == [TWO_LAUNCH, 0, 0]
    for s in range(m):
        xo, ito, reso = orc.svl_cg(b[s], *dims, iters=9, end_res=0.0)
        assert it[s] == ito and abs(res[s] - reso) <= 1e-4 * reso
        assert np.max(np.abs(x[s] - xo)) <= 1e-4 * np.max(np.abs(xo))


def test_waits_are_bounded(gc, dev):
    d = torch.zeros(64, dtype=torch.float32, device=dev)
    for first, others in ((1e9, 0.0), (0.0, float("inf")), (float("nan"), 0.0)):
        assert gc.lib.gpucad_svl_cg_form(gc.ptr(d), 1, 4, 4, 4, 4, 0.0, 0, first, others, None,
                                         None, None) == gc.E_ARG
    for m, form in ((0, 0), (5, 0), (1, 3), (1, -1)):
        assert gc.lib.gpucad_svl_cg_form(gc.ptr(d), m, 4, 4, 4, 4, 0.0, form, 0.0, 0.0, None, None,
                                         None) == gc.E_ARG


def test_a_solve_that_gave_up_is_not_tried_at_once(gc, orc, dev):
    dims = (40, 24, 40)
    b = rhs(orc, dims, 1)
    want = solve(gc, dev, b, dims, 12, 0.0, TWO_LAUNCH)
    assert solve(gc, dev, b, dims, 12, 0.0, ON_CHIP)[3][0] == ON_CHIP
    assert solve(gc, dev, b, dims, 12, 0.0)[3][0] == ON_CHIP
    assert solve(gc, dev, b, dims, 12, 0.0, 0, -1.0, -1.0)[3][0] == TWO_LAUNCH
    by = []
    for _ in range(65):  # nothing holds the CUs any more
        x, it, res, how = solve(gc, dev, b, dims, 12, 0.0)
        assert np.array_equal(x, want[0]) or how[0] == ON_CHIP
        by.append(how[0])
    assert by == [TWO_LAUNCH] * 64 + [ON_CHIP]
    # a solve on the chip that the caller asked for and that ends clears it too
    assert solve(gc, dev, b, dims, 12, 0.0, 0, -1.0, -1.0)[3][0] == TWO_LAUNCH
    assert solve(gc, dev, b, dims, 12, 0.0)[3][0] == TWO_LAUNCH
    assert solve(gc, dev, b, dims, 12, 0.0, ON_CHIP)[3][0] == ON_CHIP
    assert solve(gc, dev, b, dims, 12, 0.0)[3][0] == ON_CHIP


@pytest.mark.parametrize("dims", [(8, 6, 5), (12, 20, 40), (64, 40, 24)])
def test_the_largest_values(gc, orc, dev, dims):
    """A constant close to the type's largest value is in the operator's null
    space, so no term of it may overflow: d.q is 0 and the step infinite."""
    b = np.full((1, dims[0] * dims[1] * dims[2]), 1.125 * 2.0 ** 126, np.float32)
    with np.errstate(all="ignore"):
        xo, ito, reso = orc.svl_cg(b[0], *dims, iters=5, end_res=0.0)
    assert np.all(np.isposinf(xo)) and np.isnan(reso)
    for form in (TWO_LAUNCH, ON_CHIP):
        x, it, res, how = solve(gc, dev, b, dims, 5, 0.0, form)
        assert how[0] == form
        assert it == [ito] and np.isnan(res[0])
        assert np.array_equal(x[0], xo)


@pytest.mark.parametrize("r", [0, 2, 4])
@pytest.mark.parametrize("fine", [(1, 9, 70), (3, 70, 5), (4, 33, 9), (5, 7, 37), (8, 40, 8),
                                  (17, 5, 13), (31, 8, 8), (64, 3, 5), (65, 6, 7), (127, 9, 2),
                                  (128, 3, 11), (129, 3, 11), (256, 2, 5), (1030, 2, 3),
                                  (40000, 1, 2)], ids=lambda f: "x".join(map(str, f)))
def test_synthesis_rows(gc, orc, dev, fine, r):
    """Fine rows of every share of a wave and longer than several, against the
    same points of a synthesis that has them in the middle of longer rows:
    the same taps and arithmetic, so the same bits."""
    c = np.random.default_rng(23).standard_normal(((2 * r + 1) ** 3, 2)).astype(np.float32)

    def run(fx):
        p = gc.svl_params(9, lattice_type="b", const_period=7.0, range_=r, cg_max_iter=12,
                          harmonics=(2 * r + 1) ** 3, cg_end_res=1e-6)
        p.ny, p.nz, p.fx, p.fy, p.fz = 6, 5, fx, fine[1], fine[2]
        p.fine_dx = 8.0 / fine[0]
        svl, _ = gc.svl_field(p, torch.from_numpy(c).to(dev))
        return svl.cpu().numpy().reshape(fine[2], fine[1], fx), p

    got, p = run(fine[0])
    longer, _ = run(fine[0] + 300)
    assert np.array_equal(got.view(np.uint32), longer[:, :, :fine[0]].copy().view(np.uint32))
    if fine[0] <= 256:
        ref, _, _ = orc.svl_field(p, c, None)
        assert np.max(np.abs(got.reshape(-1) - ref)) < 2e-2 * max(1e-3, np.max(np.abs(ref)))
