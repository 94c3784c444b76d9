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


def fwht(v):
    """quant.rs:109-115 in f32, the butterflies in the kernels' order."""
    v, h = v.astype(np.float32), 1
    while h < 128:
        w = v.reshape(-1, 2, h)
        v = np.stack([w[:, 0] + w[:, 1], w[:, 0] - w[:, 1]], axis=1).reshape(-1)
        h *= 2
    return v * np.uint32(0x3db504f3).view(np.float32)


def a8(x, bits):
    """A group's codes in act_pos order and its scale: the greatest magnitude
    that is a number over 127, or 1 where p and p + 64 both hold a NaN."""
    y = fwht(x)
    n = np.isnan(y)
    m = np.float32(0) if (n & np.roll(n, 64)).any() or n.all() else np.abs(y[~n]).max()
    s = m * np.uint32(0x3c010204).view(np.float32) if m > 0 else np.float32(1)
    r = y * (np.float32(1) / s)
    t = np.trunc(r)
    t = np.where(np.abs(r - t) >= 0.5, t + np.copysign(np.float32(1), r), t)  # half away from zero
    code = np.where(np.isnan(r), -128, np.clip(np.where(np.isnan(t), r, t), -128, 127)).astype(np.int8)
    p, out = np.arange(128), np.empty(128, np.int8)
    out[(p % 4) * 32 + p // 4 if bits == 2 else (p % 2) * 64 + p // 2] = code
    return out, s


@pytest.mark.parametrize("bits", [4, 2])
def test_groups_holding_nan(nh, bits):
    """Where the rotation leaves NaNs: the scale is 1 for one at both p and
    p + 64, whatever the other positions hold; in every form of the call."""
    big = np.float32(2e38)
    x = o.seeded_normals([16 * 128], seed=6)[0].reshape(16, 128)
    x[0, 3] = np.inf                                  # infinities only
    x[1, 1] = np.nan                                  # NaN everywhere
    x[2, 0:2] = np.inf                                # infinities and NaN, the NaN in pairs
    x[3, [0, 64]] = np.inf                            # NaN at p + 64 only
    x[5, [7, 71]] = [np.inf, -np.inf]                 # NaN at p only
    # (apart from the infinities: eight groups share a wavefront)
    x[12] = 0                                         # overflow inside: NaN pairs beside finite values
    x[12, [0, 16, 32, 48, 64, 80]] = big
    x[12, [96, 112]] = -big
    x[12, 16] = np.float32(1.9e38)
    with np.errstate(all="ignore"):
        want = [a8(g, bits) for g in x]
        y = np.isnan(fwht(x[12]))
    assert y.sum() == 64 and (y == np.roll(y, 64)).all() and want[12][1] == 1
    assert np.flatnonzero([np.isinf(w[1]) for w in want]).tolist() == [0, 3, 5]
    say(f"groups holding NaN, {bits} bits")
    codes, scales = nh.QAct.new(torch.from_numpy(x.reshape(-1)).cuda(), 1, 2048, bits).download()
    assert np.array_equal(np.asarray(scales).ravel().view(np.uint32), np.array([w[1] for w in want]).view(np.uint32))
    assert np.array_equal(np.asarray(codes).reshape(16, 128), np.stack([w[0] for w in want]))


def test_one_row_product_of_overflowing_input(nh):
    """The one-launch product does its own A8: the same groups as the two steps."""
    x = np.zeros(256, np.float32)
    x[[0, 32, 48, 64, 80]], x[16], x[[96, 112]] = 2e38, 1.9e38, -2e38
    x[128:] = o.seeded_normals([128], seed=7)[0]
    w = (o.seeded_normals([32 * 256], seed=8)[0] * np.float32(0.02)).astype(np.float32)
    lin = nh.QLinear([nh.QMat.from_f32(w, 32, 256)])
    xd = torch.from_numpy(x).cuda()
    say("one row that overflows in the rotation")
    one, two = lin.apply(xd, 1), lin.matmul(nh.QAct.new(xd, 1, 256, 4))
    assert torch.equal(one.view(torch.int32), two.view(torch.int32))
