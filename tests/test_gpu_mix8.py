"""GPU: the layer kernel's mix8 passes on the f32 matrix cores against the
oracle's fma chains (infer.rs:2343-2380), bit for bit: ordinary operands, a
wide range of exponents with cancellation, signed zeros, subnormal operands,
products and sums, results that overflow, infinities and NaN."""
import sys

import numpy as np
import pytest
import torch

import oracle as o
from oracle import forward

pytestmark = pytest.mark.gpu


def chains(factor, x):
    """(factor^T x, x factor) by the oracle's fma chains."""
    f = factor.astype(np.float32)
    yt, yn = np.empty((32, 32), np.float32), np.empty((32, 32), np.float32)
    lib = forward._lib()
    xt = np.ascontiguousarray(x.T)
    lib.nf_mix8(0, o._p(f), 0, o._p(x), 0, o._p(yt), 16)
    lib.nf_mix8(0, o._p(xt), 0, o._p(f), 0, o._p(yn), 16)
    return yt, yn


def operands(kind, rng):
    f = rng.standard_normal((32, 32))
    x = rng.standard_normal((32, 32))
    sign = lambda: rng.choice([-1.0, 1.0], (32, 32))
    if kind == "wide":  # sums that cancel over 2^-60 .. 2^60
        f, x = sign() * 2.0 ** rng.integers(-14, 15, (32, 32)), x * 2.0 ** rng.integers(-60, 60, (32, 32))
    elif kind == "zeros":
        f, x = f * rng.integers(0, 2, (32, 32)) * sign(), x * rng.integers(0, 2, (32, 32)) * sign()
    elif kind == "subnormal factor":
        f = sign() * rng.integers(0, 1024, (32, 32)) * 2.0 ** -24
    elif kind == "subnormal x":  # subnormal operands and products
        x = sign() * rng.integers(0, 1 << 23, (32, 32)) * 2.0 ** -149
    elif kind == "subnormal sums":
        f, x = sign() * 2.0 ** rng.integers(-24, 0, (32, 32)), x * 2.0 ** rng.integers(-140, -120, (32, 32))
    elif kind == "overflow":
        f, x = sign() * 6e4, x * 2.0 ** rng.integers(104, 112, (32, 32))
    x = x.astype(np.float32)
    if kind == "not finite":
        x[3, 5], x[9, 5], x[20, 30], x[31, 0] = np.inf, -np.inf, np.nan, np.inf
    return f.astype(np.float16), x


@pytest.mark.parametrize("kind", ["normal", "wide", "zeros", "subnormal factor", "subnormal x", "subnormal sums",
                                  "overflow", "not finite"])
def test_passes(nh, kind):
    print(f"mix8 passes: {kind}", flush=True)
    sys.stdout.flush()
    for seed in range(8):
        f, x = operands(kind, np.random.default_rng(seed))
        with np.errstate(all="ignore"):
            want = chains(f, x)
        got = nh.debug_mix8(torch.from_numpy(f).cuda(), torch.from_numpy(x).cuda())
        for g, w in zip(got, want):
            g = g.cpu().numpy()
            nan = np.isnan(w)
            assert np.array_equal(np.isnan(g), nan)
            assert np.array_equal(g.view(np.uint32)[~nan], w.view(np.uint32)[~nan])
            if kind in ("overflow", "not finite"):
                assert np.isinf(w).any()
            if kind.startswith("subnormal x"):
                assert (np.abs(w) < 2.0 ** -126).any()
