"""GPU: QMat.from_f32 (cq_pack and the tiling on the device) against from_cq of
its own download (the host's tiling) at row counts and widths inside a tile,
a panel and a group: the same products (decode and prefill), rows and bytes."""
import sys

import numpy as np
import pytest
import torch

import oracle as o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 65, 300])
@pytest.mark.parametrize("k", [1, 100, 128, 300, 4096])
def test_from_f32(nh, n, k):
    print(f"from_f32 {n} x {k}", flush=True)
    sys.stdout.flush()
    w = (o.seeded_normals([n * k], seed=n + k)[0] * np.float32(0.02)).astype(np.float32)
    m = nh.QMat.from_f32(w, n, k)
    packed, norms = m.download()
    want_p, want_n = o.cq_pack(w, k)
    assert np.array_equal(packed.ravel(), np.asarray(want_p).ravel())
    assert np.array_equal(norms.ravel(), np.asarray(want_n).ravel())
    h = nh.QMat.from_cq(packed, norms, n, k)
    for rows in (1, 5, 70):
        x = torch.from_numpy(o.seeded_normals([rows * k], seed=rows)[0]).cuda()
        a = nh.QAct.new(x, rows, k)
        assert torch.equal(m.matmul(a).view(torch.int32), h.matmul(a).view(torch.int32))
    ids = torch.tensor([0, n - 1], dtype=torch.int32, device="cuda")
    assert torch.equal(m.rows(ids).view(torch.int32), h.rows(ids).view(torch.int32))
