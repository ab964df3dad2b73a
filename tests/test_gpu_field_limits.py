"""Field launches at the limits of a launch's shape: rows as long as a launch's
first dimension holds in the order that takes eight workgroups per brick, and
more rows than its second holds, which are refused whatever the order."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def params(gc, n):
    from gpucadforam_amd import configs as CF
    return CF.make(*n, gc.TPMS_SCHWARZ_P, 64.0, sheet=False)


@pytest.mark.parametrize("nx", [(1 << 27) - 127, (1 << 27) + 1], ids=["2^27 - 127", "2^27 + 1"])
def test_longest_rows(gc, dev, nx):
    p = params(gc, (nx, 2, 2))
    f = torch.full((4 * nx,), float("nan"), dtype=torch.float32, device=dev)
    s = torch.full((gc.sign_words(nx, 2, 2),), -1, dtype=torch.int64, device=dev)
    gc.lattice_field(p, out=f, signs=s)
    assert bool((f.abs() <= 3.0).all())  # (no NaN is left)
    # the last words of each row are the ballot of the stored values
    tail = nx % 64 + 64
    rows, words = f.view(4, nx)[:, -tail:], s.view(4, -1)[:, -2:]
    bits = (rows < 0).cpu().numpy()
    for r in range(4):
        w = words[r].cpu().numpy().view(np.uint64)
        got = [(int(w[i // 64]) >> (i % 64)) & 1 for i in range(tail)]
        assert got == bits[r].astype(int).tolist()
        assert int(w[1]) >> (nx % 64) == 0


@pytest.mark.parametrize("nx", [64, 66])
def test_too_many_rows(gc, dev, nx):
    f = torch.zeros(nx * 262144 * 2, dtype=torch.float32, device=dev)
    assert gc.lib.gpucad_lattice_field(params(gc, (nx, 262140, 2)), gc.ptr(f), None, 0.0,
                                       gc.stream_handle()) == gc.OK
    torch.cuda.synchronize()
    assert gc.lib.gpucad_lattice_field(params(gc, (nx, 262144, 2)), gc.ptr(f), None, 0.0,
                                       gc.stream_handle()) == gc.E_ARG
