"""GPU: QLinear.apply (qlinear.rs:555-557) in its three forms - one f32 token
through the product that does its own A8 (small matrices), the two steps
over a caller's workspace, and the call that stages by itself - against
QAct + matmul on the same inputs, bit for bit, over the group counts of every
launch shape, widths that end inside a group, and every code width."""
import ctypes as C
import sys

import numpy as np
import pytest
import torch

import oracle as o

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def linear(nh, n, k, bits, seed):
    groups = (k + 127) // 128
    rng = np.random.default_rng(seed)
    packed = rng.integers(0, 256, (n, groups * (64 if bits == 4 else 32)), dtype=np.uint8)
    norms = (0.2 + rng.random((n, groups))).astype(np.float16).view(np.uint16)
    return nh.QLinear([nh.QMat.from_cq(packed, norms, n, k, bits)])


def two_steps(nh, lin, x, rows):
    a = nh.QAct.new(x, rows, lin.in_dim, lin.act_bits())
    return lin.matmul(a)


def bits(t):
    return t.cpu().numpy().view(np.uint32)


@pytest.mark.parametrize("k", [1, 127, 128, 200, 384, 500, 768, 1000, 1536, 2048, 3000, 4096])
@pytest.mark.parametrize("width", [4, 2, 5])
def test_one_row(nh, k, width):
    for n in (1, 16, 500):
        lin = linear(nh, n, k, width, seed=k * 7 + n)
        x = torch.from_numpy(o.seeded_normals([k], seed=k + n)[0]).cuda()
        if n == 16:
            x[: k // 2] = 0.0  # whole groups of zeros take scale 1
        say(f"one row: {n} x {k}, {width} bits, workspace {nh._lib.nh_qlinear_apply_ws_bytes(lin.fused.h, 1)}")
        want = bits(two_steps(nh, lin, x, 1))
        assert np.array_equal(bits(lin.apply(x, 1)), want)
        y = torch.empty((1, n), device="cuda")
        assert np.array_equal(bits(lin.apply_static(x, 1, y)), want)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        z = lin.apply(x, 1, stream=side)
        side.synchronize()
        assert np.array_equal(bits(z), want)


@pytest.mark.parametrize("n,k", [(8192, 4096), (8208, 4096)])
def test_one_row_large(nh, n, k):
    lin = linear(nh, n, k, 4, seed=3)
    # the last size of the one-launch form, the first of the two steps
    assert (nh._lib.nh_qlinear_apply_ws_bytes(lin.fused.h, 1) > 0) == (n > 8192)
    x = torch.from_numpy(o.seeded_normals([k], seed=4)[0]).cuda()
    assert np.array_equal(bits(lin.apply(x, 1)), bits(two_steps(nh, lin, x, 1)))


@pytest.mark.parametrize("rows", [2, 5, 64, 65, 130])
def test_rows(nh, rows):
    lin = linear(nh, 300, 500, 4, seed=rows)
    x = torch.from_numpy(o.seeded_normals([rows * 500], seed=rows)[0]).cuda()
    want = bits(two_steps(nh, lin, x, rows))
    assert np.array_equal(bits(lin.apply(x, rows)), want)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    y = lin.apply(x, rows, stream=side)
    side.synchronize()
    assert np.array_equal(bits(y), want)


def test_captured(nh):
    lin = linear(nh, 300, 500, 4, seed=9)
    for rows in (1, 7):
        x = torch.from_numpy(o.seeded_normals([rows * 500], seed=rows)[0]).cuda()
        want = bits(lin.apply(x, rows))
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            y = lin.apply(x, rows)
        for _ in range(3):
            y.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert np.array_equal(bits(y), want)


def test_in_place_and_refusals(nh):
    say("a token overwritten by its own product, and the workspace checks")
    lin = linear(nh, 256, 256, 4, seed=11)
    x = torch.from_numpy(o.seeded_normals([256], seed=12)[0]).cuda()
    want = bits(lin.apply(x, 1)).ravel()
    p = C.c_void_p(x.data_ptr())
    assert nh._lib.nh_qlinear_apply(lin.fused.h, p, 1, p, None) == 0
    torch.cuda.synchronize()
    assert np.array_equal(bits(x).ravel(), want)
    y = torch.empty((3, 256), device="cuda")
    x3 = torch.zeros((3, 256), device="cuda")
    q, r = C.c_void_p(x3.data_ptr()), C.c_void_p(y.data_ptr())
    assert nh._lib.nh_qlinear_apply_ws(lin.fused.h, q, 3, r, None, 0, None) < 0
    ws = torch.empty(nh._lib.nh_qlinear_apply_ws_bytes(lin.fused.h, 3), dtype=torch.uint8, device="cuda")
    assert nh._lib.nh_qlinear_apply_ws(lin.fused.h, q, 3, r, C.c_void_p(ws.data_ptr()), ws.numel() - 1, None) < 0
    assert nh._lib.nh_qlinear_apply_ws_bytes(None, 3) < 0
    with pytest.raises(nh.NeedleHipError, match="null argument|no rows"):
        lin.apply(x3, 0)
    torch.cuda.synchronize()
