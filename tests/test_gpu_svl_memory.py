"""What the synthesis entry points keep of device memory after a call, and the
unit cell's spectrum in pieces of its rows."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

MB = 1 << 20


def kept_by(gc, call):
    """Bytes of device memory that are taken after `call` and were not before."""
    torch.cuda.empty_cache()
    gc.check(gc.lib.gpucad_shutdown())
    gc.init(0)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    call()
    torch.cuda.synchronize()
    return before - torch.cuda.mem_get_info()[0]


@pytest.mark.parametrize("n", [100, 170], ids=["on the chip", "two launches"])
def test_synthesis_keeps_five_vectors(gc, dev, n):
    """Five vectors of the three solves, in an arena a quarter larger than asked
    (the right-hand sides are one of the five)."""
    p = gc.svl_params(n, lattice_type="b", const_period=9.0, range_=1, harmonics=27, cg_max_iter=4)
    p.fx, p.fy, p.fz = 16, 16, 16
    c = torch.zeros(27, dtype=torch.complex64, device=dev)
    gc.svl_field(p, c)  # (torch's own pools)
    kept = kept_by(gc, lambda: gc.svl_field(p, c))
    assert kept <= 1.25 * 5 * 3 * n ** 3 * 4 + 16 * MB, kept / MB


def test_spectrum_keeps_a_piece(gc, dev):
    ny = nz = 2000
    cell = torch.zeros(ny * nz, dtype=torch.float32, device=dev)
    out = torch.zeros(125, dtype=torch.complex64, device=dev)
    kept = kept_by(gc, lambda: gc.check(gc.lib.gpucad_unit_spectrum(gc.ptr(cell), 1, ny, nz, 2,
                                                                    gc.ptr(out))))
    assert kept <= 32 * MB, kept / MB


@pytest.mark.parametrize("dims,r", [((1, 512, 512), 1), ((1, 512, 513), 2), ((2, 700, 750), 4),
                                    ((5, 1024, 513), 1)])
def test_spectrum_of_many_rows(gc, dev, dims, r):
    """As many rows as are held at a time, one slab more, twice as many and more
    (FP64 sums, one rounding to FP32: 1e-6 of the largest coefficient)."""
    nx, ny, nz = dims
    cell = np.random.default_rng(24).standard_normal(nx * ny * nz).astype(np.float32)
    side = 2 * r + 1
    out = torch.zeros(side ** 3, dtype=torch.complex64, device=dev)
    gc.check(gc.lib.gpucad_unit_spectrum(gc.ptr(torch.from_numpy(cell).to(dev)), nx, ny, nz, r,
                                         gc.ptr(out)))
    f = np.fft.fftn(cell.reshape(nz, ny, nx).astype(np.float64)) / (nx * ny * nz)
    k = np.arange(-r, r + 1)
    ref = f[np.ix_(k % nz, k % ny, k % nx)].reshape(-1)
    assert np.max(np.abs(out.cpu().numpy() - ref)) < 1e-6 * np.max(np.abs(ref))
