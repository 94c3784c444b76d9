"""GPU: what sessions hold on the device, and feeds of more rows than a
session's own buffers have, which a model's sessions run through one set of
buffers: several sessions on streams and threads of their own, a set that
grows while feeds are queued, clones, and the memory given back."""
import sys
import threading

import numpy as np
import pytest
import torch

import oracle as o
from oracle import cact, forward
from test_gpu_session import archive

pytestmark = pytest.mark.gpu

G = cact.Geometry(vocab=300, num_layers=2, engram_slots=64, engram_sites=(1,), global_layers=(0,), sliding_window=300)


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def model(nh):
    return nh.Model.from_archive(archive(G, seed=141))


def row_bytes(g, chunks):
    d, sites, heads = g.d_model, len(g.engram_sites), g.num_heads
    nq = heads * g.qk_head_dim + g.num_kv_heads * (g.qk_head_dim + g.v_head_dim) + heads * g.v_head_dim
    floats = 8 * d + 64 + nq + heads * g.qk_head_dim + sites * 3 * d + g.qk_head_dim
    return 4 * (floats + heads * chunks * (g.v_head_dim + 2)) + (2 + sites) * (d + 128) * 33 // 32 + 1


def free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_sessions_share_the_longest_feeds_rows(nh):
    cap, n = 4096, 6
    start = free()
    model = nh.Model.from_archive(archive(G, seed=142))
    state = cap * G.num_layers * G.num_kv_heads * (G.qk_head_dim + G.v_head_dim + 8) + \
        2048 * G.num_layers * G.num_kv_heads * (G.qk_head_dim + G.v_head_dim + 8) + \
        len(G.engram_sites) * cap * (G.d_model + G.d_model // 8)
    before = free()
    first = model.session(cap)
    held = free()
    rest = [model.session(cap) for _ in range(n - 2)] + [first.clone()]
    each = (held - free()) / (n - 1)
    bound = state + 513 * row_bytes(G, cap // 256) + (8 << 20)
    say(f"a session of {cap} positions: {each / 1e6:.1f} MB, the first {(before - held) / 1e6:.1f}; bound {bound / 1e6:.1f}")
    assert each <= bound
    wide = 2048 * row_bytes(G, cap // 256) + (8 << 20)
    assert before - held <= bound + wide
    del first, rest
    assert before - free() <= wide  # (the model keeps them for its next session)
    del model
    # (the code objects and small blocks the runtime loaded meanwhile stay)
    assert start - free() <= 32 << 20 < wide // 4


def feeds(s, sizes, seed, stream=None):
    return [s.forward(o.random_tokens(n, 300, seed=seed + i), forward.OUT_LAST_LOGITS, stream=stream)
            for i, n in enumerate(sizes)]


def same(a, b):
    return all(torch.equal(x.view(torch.int32), y.view(torch.int32)) for x, y in zip(a, b, strict=True)) and \
        all(bool(torch.isfinite(x).all()) for x in a)


SIZES = (1100, 1, 40, 700)


def test_streams_take_turns(nh, model):
    say("three sessions' long feeds on three streams, the third's buffers grown while the others are queued")
    want = [feeds(model.session(1900 + 700 * i), SIZES, 150 + 10 * i) for i in range(3)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(3)]
    for _ in range(3):
        s = [model.session(1900), model.session(2600)]
        got = [feeds(s[0], SIZES[:2], 150, streams[0]), feeds(s[1], SIZES, 160, streams[1])]
        got[0] += [s[0].forward(o.random_tokens(n, 300, seed=152 + i), forward.OUT_LAST_LOGITS, stream=streams[0])
                   for i, n in enumerate(SIZES[2:])]
        third = model.session(3300)
        got.append(feeds(third, SIZES, 170, streams[2]))
        torch.cuda.synchronize()
        for g, w in zip(got, want):
            assert same(g, w)


def test_threads(nh, model):
    say("two threads, a session and a stream each")
    want = [feeds(model.session(1900), SIZES, 180 + 10 * i) for i in range(2)]
    torch.cuda.synchronize()
    got, errors = [None, None], []

    def work(i):
        try:
            st = torch.cuda.Stream()
            for _ in range(3):
                got[i] = feeds(model.session(1900), SIZES, 180 + 10 * i, st)
                st.synchronize()
        except Exception as e:  # reported below, in the test's own thread
            errors.append(e)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not errors, errors
    assert same(got[0], want[0]) and same(got[1], want[1])


def test_clone_after_a_long_feed(nh, model):
    say("a clone carries on as its source does")
    s = model.session(2600)
    feeds(s, (1300,), 200)
    c = s.clone()
    a, b = feeds(s, (700, 1, 33), 210), feeds(c, (700, 1, 33), 210)
    assert same(a, b)
    assert np.array_equal(s.generate_greedy(4)[0], c.generate_greedy(4)[0])


def test_captured_long_feed(nh, model):
    """A captured feed keeps to the session's own rows: replayed beside other
    sessions' long feeds it gives what the eager feed gave."""
    say("a captured feed of 1100 tokens")
    toks = o.random_tokens(1100, 300, seed=220)
    s, other = model.session(1900), model.session(1900)
    want = s.forward(toks, forward.OUT_ALL_LOGITS).clone()
    torch.cuda.synchronize()
    s.reset()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = s.forward(toks, forward.OUT_ALL_LOGITS)
    beside = feeds(other, SIZES, 230)
    for _ in range(3):
        y.zero_()
        other.reset()
        st = torch.cuda.Stream()
        again = feeds(other, SIZES, 230, st)
        g.replay()
        torch.cuda.synchronize()
        assert same([y], [want]) and same(again, beside)
