"""One-grid field launches in the order that puts a row's bricks on one XCD
(16 M points and more, rows that end inside a line when rotated): every point
and sign word is written by some workgroup, with rows of bricks that do and do
not fill groups of eight, against the oracle on slabs of planes."""
import math

import numpy as np
import pytest
import torch

from helpers import to_np, ulp_diff
from test_gpu_lattice import FIELD_ULP

pytestmark = pytest.mark.gpu

GRIDS = [("plain", (299, 250, 230)), ("plain", (256, 252, 261)), ("rot", (299, 250, 230)),
         ("rot", (1030, 17, 961)), ("bent", (97, 601, 290)), ("plain", (2050, 3, 2731))]


@pytest.mark.parametrize("form,n", GRIDS, ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
def test_field_in_xcd_order(gc, orc, dev, form, n):
    from gpucadforam_amd import configs as CF
    p = CF.make(*n, gc.TPMS_GYROID, 21.0, 33.0 if form == "rot" else 21.0, rot0=0.0,
                rot1=math.pi / 2 if form == "rot" else 0.0,
                bend_radius=2.0 if form == "bent" else 0.0, sheet=True, t0=0.3,
                prim=gc.PRIM_SPHERE, op=gc.OP_INTERSECT, center=(0.5, 0.5, 0.5), radius=0.45,
                half=(0.4, 0.4, 0.4))
    f = torch.full((p.npoints(),), float("nan"), dtype=torch.float32, device=dev)
    words = gc.sign_words(*n)
    s = torch.full((words,), -1, dtype=torch.int64, device=dev)
    gc.lattice_field(p, out=f, signs=s)
    assert not torch.isnan(f).any()
    plane, wplane = n[0] * n[1], words // n[2]
    for z0 in (0, n[2] // 2 - 1, n[2] - 3):
        z1 = z0 + 3
        got = to_np(f[z0 * plane:z1 * plane])
        ref = orc.lattice_field_f32(p, z0, z1)
        assert ulp_diff(got, ref).max() <= FIELD_ULP
    # every sign word is the ballot of the stored values
    for z0 in range(0, n[2], 64):
        z1 = min(z0 + 64, n[2])
        got = to_np(f[z0 * plane:z1 * plane])
        sref = orc.signs(got, n[0], n[1], z1 - z0, 0.0)
        assert np.array_equal(to_np(s[z0 * wplane:z1 * wplane]).view(np.uint64), sref)
