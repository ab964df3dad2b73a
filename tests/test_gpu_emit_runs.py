"""Mesh emission where its launch shape changes: exactly as many blocks as are
summed without a scan, and workgroups in runs per XCD with rows of several
words, in chunks of 16 and of 32 words and not filling their last run."""
import ctypes as C

import numpy as np
import pytest
import torch

from test_gpu_emit import _args, _field

pytestmark = pytest.mark.gpu

SHAPES = [(64, 256, 512),   # 512 blocks
          (130, 300, 480),  # 1688 blocks, rows of 3 words: chunks of 16 words, runs of 4 blocks
          (70, 640, 829)]   # 4145 blocks, rows of 2 words: chunks of 32 words, runs of 8 blocks


@pytest.mark.parametrize("n", SHAPES, ids=lambda n: "x".join(map(str, n)))
def test_emit_matches_oracle(gc, orc, dev, n):
    field = _field(n, "smooth", 1)
    v_ref, t_ref, _ = orc.extract_indexed(field, *n, spacing=(1, 1, 1))
    nv, nt = len(v_ref), len(t_ref)
    f = torch.from_numpy(field).to(dev)
    ws = torch.empty(gc.extract_workspace_bytes(*n), dtype=torch.uint8, device=dev)
    counts = torch.zeros(2, dtype=torch.int64, device=dev)
    v = torch.full((nv, 3), -7.0, dtype=torch.float32, device=dev)
    t = torch.full((nt, 3), -7, dtype=torch.int32, device=dev)
    a = _args(gc, f, n, v, nv, t, nt, ws, counts)
    gc.check(gc.lib.gpucad_extract(C.byref(a), None, gc.stream_handle()))
    assert counts.tolist() == [nv, nt]
    assert np.array_equal(v.cpu().numpy().view(np.uint32), v_ref.view(np.uint32))
    assert np.array_equal(t.cpu().numpy(), t_ref.astype(np.int32))
