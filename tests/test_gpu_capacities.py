"""GPU: sessions of very large capacities give what a small one gives, bit for
bit, around the strides their cache takes (grouped attention from 64,993
positions on, where the staging slots make the value stride 65,536 or more),
causal and under a span."""
import sys

import numpy as np
import pytest

import oracle as o
from oracle import cact, forward
from test_gpu_session import archive

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap", [64992, 64993, 65520, 70000, 300000])
def test_large_capacity(nh, cap):
    print(f"capacity {cap}", flush=True)
    sys.stdout.flush()
    g = cact.Geometry(vocab=300, num_layers=2, engram_slots=64, engram_sites=(1,), global_layers=(0,), sliding_window=48)
    m = nh.Model.from_archive(archive(g, seed=131))
    small, large = m.session(400), m.session(cap)
    for span in (None, (20, 64)):
        outs = []
        for s in (small, large):
            s.reset()
            if span:
                s.set_attend(*span)
            got = [s.forward(o.random_tokens(n, 300, seed=132 + n), forward.OUT_LAST_LOGITS).cpu().numpy()
                   for n in (290, 1, 65)]
            outs.append(np.concatenate(got))
        assert np.isfinite(outs[0]).all()
        assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
