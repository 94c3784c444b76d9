"""GPU: A8 of f32 rows (QAct::new, with and without the fused RMSNorm) against
the oracle where its lanes, wavefronts and workgroups end: widths inside a
lane's 16 positions and a group, rows around a workgroup's four, unaligned
rows and scales, both activation orders; and groups holding infinities or
NaN, which must not disturb their neighbours."""
import sys

import numpy as np
import pytest
import torch

import oracle as o

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("bits", [4, 2])
@pytest.mark.parametrize("k", [1, 15, 17, 127, 128, 130, 1000, 4096])
def test_rows(nh, k, bits):
    for rows in (1, 2, 9):
        say(f"A8 of {rows} x {k}, {bits} bits")
        x = o.seeded_normals([rows * k], seed=k + rows)[0]
        a = o.OQAct.new(x, rows, k, bits)
        want = a.xq, a.sx
        buf = torch.zeros(rows * k + 1, device="cuda")
        for off in (0, 1):  # 16-byte aligned rows, then not
            buf[off:off + rows * k] = torch.from_numpy(x).cuda()
            got = nh.QAct.new(buf[off:off + rows * k], rows, k, bits).download()
            for g, w in zip(got, want):
                assert np.array_equal(np.asarray(g).reshape(-1).view(np.uint8), np.asarray(w).reshape(-1).view(np.uint8))


@pytest.mark.parametrize("bits", [4, 2])
@pytest.mark.parametrize("k", [16, 112, 768, 2048, 2064, 4096])
def test_norm_rows(nh, k, bits):
    for rows in (1, 3, 4, 5, 8):
        say(f"norm and A8 of {rows} x {k}, {bits} bits")
        x = (o.seeded_normals([rows * k], seed=k + rows)[0] * np.float32(3)).astype(np.float32)
        s = (0.1 * o.seeded_normals([k], seed=k)[0]).astype(np.float16)
        h = np.concatenate([o.zcn16(x[i * k:(i + 1) * k], s.view(np.uint16)) for i in range(rows)])
        a = o.OQAct.new(h, rows, k, bits)
        want = a.xq, a.sx
        sb = torch.zeros(k + 1, dtype=torch.float16, device="cuda")
        for off in (0, 1):
            sb[off:off + k] = torch.from_numpy(s).cuda()
            got = nh.QAct.new(torch.from_numpy(x).cuda(), rows, k, bits, norm_scale=sb[off:off + k]).download()
            for g, w in zip(got, want):
                assert np.array_equal(np.asarray(g).reshape(-1).view(np.uint8), np.asarray(w).reshape(-1).view(np.uint8))


def test_not_finite(nh):
    k, rows = 1024, 3
    x = o.seeded_normals([rows * k], seed=5)[0]
    clean = nh.QAct.new(torch.from_numpy(x).cuda(), rows, k, 4).download()
    y = x.copy()
    y[3] = np.inf                # a group of infinities
    y[128 + 1] = np.nan          # a group of NaN
    y[256:258] = np.inf          # infinities and NaN
    got = nh.QAct.new(torch.from_numpy(y).cuda(), rows, k, 4).download()
    gx, gs = np.asarray(got[0]).reshape(rows, 8, 128), np.asarray(got[1]).reshape(rows, 8)
    cx, cs = np.asarray(clean[0]).reshape(rows, 8, 128), np.asarray(clean[1]).reshape(rows, 8)
    assert np.array_equal(gx[0, 3:], cx[0, 3:]) and np.array_equal(gx[1:], cx[1:])
    assert np.array_equal(gs[0, 3:], cs[0, 3:]) and np.array_equal(gs[1:], cs[1:])
    assert np.isinf(gs[0, 0]) and (gx[0, 0] == -128).all()   # inf * (1 / inf) is NaN
    assert gs[0, 1] == 1.0 and (gx[0, 1] == -128).all()
