"""GPU: feeds of several chunks under an attention span, fed together with
their keys staged beside the ring, against the oracle feeding them chunk by
chunk: sinks inside, at and past a chunk's edge, a ring as long as a chunk,
one that wraps within a feed and one that never fills, odd feeds (whose row
pairs straddle chunks), and stale positions (which take the chunked form)."""
import sys

import pytest

import oracle as o
from oracle import cact, forward
from test_gpu_session import Pair, archive

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("sink,ring,window", [(0, 32, 8), (37, 96, 0), (64, 64, 64), (5, 300, 48), (130, 33, 20)])
def test_feeds(nh, sink, ring, window):
    say(f"staged feeds: sink {sink}, ring {ring}, window {window}")
    g = cact.Geometry(vocab=300, num_layers=2, engram_slots=64, engram_sites=(1,), global_layers=(0,),
                      sliding_window=window)
    p = Pair(nh, archive(g, seed=101), 420)
    p.attend(sink, ring)
    for i, n in enumerate([67, 2, 95, 1, 130]):
        p.fwd(o.random_tokens(n, 300, seed=102 + i), forward.OUT_LAST_LOGITS if i else forward.OUT_ALL_LOGITS,
              f"feed {n}")
    p.steps(o.random_tokens(2, 300, seed=110))
    p.rollback(20)  # leaves stale slots past the end
    p.fwd(o.random_tokens(70, 300, seed=111), label="after rollback")
    p.rewind_zeroed(40)
    p.prefill(o.random_tokens(66, 300, seed=112), label="after rewind")
    p.steps(o.random_tokens(2, 300, seed=113), label="tail")
    p.done(f"staged ({sink}, {ring})")
