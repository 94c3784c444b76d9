"""GPU: every position's logits of a feed (one launch with each row's decode
combine, crates/needle-engine/src/qlinear.rs:340-350) against the oracle, at
the row counts where its token tiles and launch forms change, over a head
whose rows end inside a 16-row tile."""
import sys

import numpy as np
import pytest

import oracle as o
from oracle import cact, forward
from test_gpu_session import SMALL, Pair, archive

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


# up to 16 rows: one token tile a workgroup; up to 32: two; above: four
@pytest.mark.parametrize("vocab", [300, 320])
@pytest.mark.parametrize("n", [2, 3, 15, 16, 17, 32, 34, 64, 66, 130])
def test_row_counts(nh, n, vocab):
    say(f"all logits of {n} rows, {vocab} head rows")
    p = Pair(nh, archive(cact.Geometry(**{**SMALL, "vocab": vocab}), seed=71), n + 2)
    got = p.fwd(o.random_tokens(n, vocab, seed=72 + n), forward.OUT_ALL_LOGITS)
    assert got.shape == (n, vocab)
    # the last row stays the session's logits: a greedy pick reads them
    pick = p.g.generate_greedy(1)
    assert int(np.asarray(pick[0] if isinstance(pick, tuple) else pick).ravel()[0]) == int(np.argmax(got[-1]))
    p.done(f"{n} rows")
