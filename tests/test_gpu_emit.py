"""Mesh emission at the edges of its chunks: rows that end inside, at and one
or two points past a 32-point half, launches of chunks of 8, 16 and 32 words
with and without a scan of their own, and capacities that cut the mesh off."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (31, 3, 5), (32, 5, 4), (33, 4, 6), (34, 3, 3), (63, 6, 5), (64, 9, 7),
          (65, 4, 9), (66, 5, 5), (97, 7, 131),
          (64, 255, 257),   # 256 blocks: the last one that starts with chunks of 8 words is 255
          (40, 300, 437),   # 513 blocks: one more than are summed without a scan
          (2, 1030, 1020),  # 4104 blocks: chunks of 32 words
          (129, 33, 65)]


def _field(n, kind, seed):
    rng = np.random.default_rng(seed)
    nx, ny, nz = n
    if kind == "noise":  # every case of the table, up to three edges per point
        return rng.standard_normal(nx * ny * nz).astype(np.float32)
    z, y, x = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    f = np.sin(0.31 * x) + np.cos(0.27 * y) + np.sin(0.23 * z)
    return np.ascontiguousarray(f.astype(np.float32).reshape(-1))


def _args(gc, f, n, v, vcap, t, tcap, ws, counts):
    a = gc.ExtractArgs()
    a.field, a.signs = f.data_ptr(), None
    a.nx, a.ny, a.nz, a.iso = *n, 0.0
    a.origin, a.spacing = gc.Float3(0, 0, 0), gc.Float3(1, 1, 1)
    a.vertices, a.vert_capacity, a.triangles, a.tri_capacity = v.data_ptr(), vcap, t.data_ptr(), tcap
    a.workspace, a.workspace_bytes = ws.data_ptr(), ws.numel()
    a.d_counts = counts.data_ptr()
    return a


@pytest.mark.parametrize("kind", ["noise", "smooth"])
@pytest.mark.parametrize("n", SHAPES, ids=lambda n: "x".join(map(str, n)))
def test_emit_matches_oracle(gc, orc, dev, n, kind):
    field = _field(n, kind, n[0] * 7 + n[1])
    v_ref, t_ref, _ = orc.extract_indexed(field, *n, spacing=(1, 1, 1))
    f = torch.from_numpy(field).to(dev)
    nv, nt = len(v_ref), len(t_ref)
    ws = torch.empty(gc.extract_workspace_bytes(*n), dtype=torch.uint8, device=dev)
    counts = torch.zeros(2, dtype=torch.int64, device=dev)
    v_ref, t_ref = v_ref.view(np.uint32), t_ref.astype(np.uint32)
    for vcap, tcap in ((nv, nt), (nv * 5 // 7, nt * 3 // 5), (0, nt)):
        # five records before and after the buffers must stay as they are; the
        # odd offset moves the records across the line boundaries
        v = torch.full((nv + 10, 3), -7.0, dtype=torch.float32, device=dev)
        t = torch.full((nt + 10, 3), -7, dtype=torch.int32, device=dev)
        a = _args(gc, f, n, v[5:], vcap, t[5:], tcap, ws, counts)
        gc.check(gc.lib.gpucad_extract(C.byref(a), None, gc.stream_handle()))
        assert counts.tolist() == [nv, nt]
        gv, gt = v.cpu().numpy(), t.cpu().numpy()
        assert (gv[:5] == -7).all() and (gv[5 + vcap:] == -7).all()
        assert (gt[:5] == -7).all() and (gt[5 + tcap:] == -7).all()
        assert np.array_equal(gv[5:5 + vcap].view(np.uint32), v_ref[:vcap])
        assert np.array_equal(gt[5:5 + tcap].view(np.uint32), t_ref[:tcap])
