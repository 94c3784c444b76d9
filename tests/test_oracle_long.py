"""The oracle's attention over more keys than eight chunks hold
(infer.rs:1871-2007): at every count the float64 softmax of the same
dequantized keys."""
import numpy as np
import pytest

from test_oracle_pins import F, attend, exact_query, softmax_ref


@pytest.mark.parametrize("n", [2048, 2049, 2500, 4096])
@pytest.mark.parametrize("nested", [False, True])
def test_attend_long(n, nested):
    rng = np.random.default_rng(n)
    q, q8, c = exact_query(rng, 48)
    k8 = rng.integers(-128, 128, size=(n, 48)).astype(np.int8)
    ks = rng.uniform(0.03, 0.08, size=n).astype(F)
    v8 = rng.integers(-128, 128, size=(n, 64)).astype(np.int8)
    vs = rng.uniform(0.01, 0.05, size=n).astype(F)
    got = attend(k8, ks, v8, vs, q, nested)
    want = softmax_ref(q8, c, k8, ks, v8, vs)
    # (the bound of the shorter counts: the digits' steps are per chunk)
    assert np.abs(got - want).max() <= 1e-5 * 127 * float(vs.max())
