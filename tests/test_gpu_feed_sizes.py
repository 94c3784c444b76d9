"""GPU: feeds at the row counts where their launches change, against the
oracle: more rows than the chip has CUs (two rows a layer workgroup), with an
odd count (the last workgroup's second row empty), the head's rows beginning
inside a pair, cells, and the widest model; more rows than a session's own
buffers hold, at and past the longest feed, in a capacity that keeps the
smaller feeds, and under an attention span."""
import sys

import pytest
import torch

import oracle as o
from oracle import cact, forward
from test_gpu_session import Pair, archive, same

pytestmark = pytest.mark.gpu

TWO = dict(vocab=300, num_layers=2, engram_slots=64, engram_sites=(0, 1), global_layers=(0,), sliding_window=300)


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def cus():
    return torch.cuda.get_device_properties(0).multi_processor_count


def tokens(n, seed):
    return o.random_tokens(n, 300, seed=seed)


# rows past the CU count: the first odd and even counts of the two-row kernel,
# an odd one whose row pairs straddle chunks
@pytest.mark.parametrize("d", [768, 1024])
@pytest.mark.parametrize("extra", [1, 2, 3, 45])
def test_two_rows_a_workgroup(nh, d, extra):
    n = cus() + extra
    say(f"feeds of {n} rows, d_model {d}: every position's logits, the last one's with cells, hidden rows")
    data = archive(cact.Geometry(**TWO, d_model=d), seed=161)
    p = Pair(nh, data, 2 * n + 8)
    p.fwd(tokens(n, 162), forward.OUT_ALL_LOGITS, "all logits")
    p.steps(tokens(2, 163))
    p.fwd(tokens(n, 164), forward.OUT_LAST_HIDDEN, "last hidden")
    p.heads([0, 7, 299])
    q = Pair(nh, data, n + 8)
    for mode in (forward.OUT_LAST_LOGITS, forward.OUT_HIDDEN):
        q.g.reset()
        q.o = q.f.session(n + 8)
        go, gc = q.g.forward_cells(tokens(n, 165), mode)
        wo, wc = q.o.forward_cells(tokens(n, 165), mode)
        same(f"mode {mode}", go.cpu().numpy(), wo, q.stats)
        same(f"mode {mode} cells", gc.cpu().numpy(), wc, q.stats)
        q.steps(tokens(2, 166))
    p.done(f"{n} rows")
    q.done(f"{n} rows with cells")


# 1,060 rows in one launch; 2,048 + 33 (32 and a step); a capacity past 64
# attention chunks, whose feeds stay at 512 rows
@pytest.mark.parametrize("cap,n,mode", [(1100, 1060, forward.OUT_ALL_LOGITS), (2200, 2081, forward.OUT_LAST_LOGITS),
                                        (16500, 700, forward.OUT_LAST_LOGITS)])
def test_longest_feeds(nh, cap, n, mode):
    say(f"a prompt of {n} tokens in a session of {cap} positions")
    p = Pair(nh, archive(cact.Geometry(**TWO), seed=171), cap)
    p.fwd(tokens(n, 172), mode, "prompt")
    p.steps(tokens(3, 173))
    p.rollback(2)
    p.fwd(tokens(30, 174), forward.OUT_ALL_LOGITS, "a chunk")
    p.done(f"{n} in {cap}")


# staged feeds of more than a session's own rows, one that splits in two, and
# an odd one with two rows a workgroup
@pytest.mark.parametrize("sink,ring,n", [(37, 300, 700), (118, 256, 2100), (5, 90, 301)])
def test_longest_span_feeds(nh, sink, ring, n):
    say(f"{n} tokens under sink {sink}, ring {ring}")
    p = Pair(nh, archive(cact.Geometry(**TWO), seed=181), n + 200)
    p.attend(sink, ring)
    p.fwd(tokens(sink, 182), forward.OUT_NONE, "the sink")
    p.fwd(tokens(n, 183), forward.OUT_LAST_LOGITS, "prompt")
    p.steps(tokens(2, 184))
    p.fwd(tokens(66, 185), forward.OUT_ALL_LOGITS, "after")
    p.done(f"span ({sink}, {ring})")
