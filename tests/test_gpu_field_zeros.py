"""Zeros of the lattice field carry the oracle's sign: grids with points on
half periods, where the sines of a solid lattice's terms vanish (bit for bit;
the arithmetic there is exact)."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("period", [1.0, 2.0, 4.0])
@pytest.mark.parametrize("rot", [0.0, math.pi / 2], ids=["straight", "rotated"])
@pytest.mark.parametrize("tpms", ["GYROID", "SCHWARZ_P", "DIAMOND"])
@pytest.mark.parametrize("n", [(9, 9, 9), (66, 9, 10)], ids=lambda n: "x".join(map(str, n)))
def test_zero_signs(gc, orc, dev, n, tpms, rot, period):
    from gpucadforam_amd import configs as CF
    p = CF.make(*n, getattr(gc, "TPMS_" + tpms), period, period, rot0=0.0, rot1=rot, sheet=False)
    f = torch.empty(p.npoints(), dtype=torch.float32, device=dev)
    gc.lattice_field(p, out=f)
    got, ref = f.cpu().numpy(), orc.lattice_field_f32(p)
    zero = ref == 0
    assert tpms == "SCHWARZ_P" or zero.any()
    assert np.array_equal(got[zero].view(np.uint32), ref[zero].view(np.uint32))
    # the batched form evaluates the same body
    b = gc.Batch([p, p], brick_x=32, brick_lz=4, use_graph=False, vert_capacity=1 << 16,
                 tri_capacity=1 << 17)
    b.run()
    res = b.results(allow_overflow=True)
    for i in range(2):
        g = b.field(i, res).cpu().numpy()
        assert np.array_equal(g[zero].view(np.uint32), ref[zero].view(np.uint32))
