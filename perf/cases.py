"""The work a program gives this framework, as measurable cases.

A case is a dict of plain values; `prepare` makes what the program holds
before the call (packed weights, a loaded model and its session, device
inputs), `run` is one pass through the public calls of `needle_hip`, `work`
the bytes and operations that pass cannot do without, `exact` its result in
64 bits by plain torch.

Kinds:
  apply    QLinear.apply: A8 of f32 rows and the fused products, one call
  sweep    the one-token product of `count` matrices in turn, captured once as
           a HIP graph (a decoding loop's products)
  project  the fused RMSNorm and A8 of `rows` tokens, then their product
  lookup   embedding rows of a batch of ids, and the sparse head over an agent's candidates
  pack     CQ-W4 packing of an f32 matrix and its upload
  turn     a fresh session: a prompt (with a span: a static prefix, then more
           tokens), then greedy decoding on the device
  steps    single-token steps of a session that already holds a long context
  prefill  one prompt into a fresh session, the last position's logits or all
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "needle-rs_amd"))

import needle_hip as nh  # noqa: E402
from needle_hip import archive  # noqa: E402

GROUP = 128
# The published Needle 3: 8,192 rows of logits over the default geometry.
VOCAB = 8192
# q | k | v | gate of a Needle-3 layer, the fused projection of every token.
QKVG = (576, 96, 128, 768)
MAX_KEYS = 4096


def listed():
    return [
        # One token through a layer's q|k|v|gate: the smallest call a decoding
        # program makes, where launches and host time count.
        {"name": "apply_token", "kind": "apply", "rows": 1, "k": 768, "n": 1568, "bits": 4},
        # A prompt chunk's rows (not a multiple of 4) through a 2-bit matrix
        # with a ragged width and height.
        {"name": "apply_chunk_2bit", "kind": "apply", "rows": 45, "k": 3000, "n": 770, "bits": 2},
        # The benchmark's decode product over matrices that no cache holds.
        {"name": "sweep_2048x8192", "kind": "sweep", "count": 32, "k": 2048, "n": 8192, "bits": 4},
        # The prefill projection at the benchmark's largest token count.
        {"name": "project_1024", "kind": "project", "rows": 1024, "k": 768, "n": 3072, "bits": 4},
        # Every position of a long prompt against the head (scoring a prompt).
        {"name": "score_head", "kind": "project", "rows": 4096, "k": 768, "n": 8192, "bits": 4},
        # Packing and uploading a projection's f32 weights.
        {"name": "pack", "kind": "pack", "n": 3072, "k": 768},
        # A short conversation turn without a span: 118 tokens in, 32 out.
        {"name": "turn", "kind": "turn", "prompt": 118, "fill": 0, "ring": 0, "steps": 32},
        # The agent's turn: its static prefix as the sink, 300 more tokens,
        # 32 greedy tokens under its KV window of 256.
        {"name": "turn_agent", "kind": "turn", "prompt": 118, "fill": 300, "ring": 256, "steps": 32},
        # Steps late in a long conversation, every key visible to the global layers.
        {"name": "steps_long", "kind": "steps", "context": 2900, "steps": 8},
        # The benchmark's prefill: one 512-token sequence.
        {"name": "prefill_512", "kind": "prefill", "tokens": 512, "outputs": "last"},
        # Scoring a sequence: the logits of every position.
        {"name": "prefill_all", "kind": "prefill", "tokens": 300, "outputs": "all"},
        # A document in the prompt.
        {"name": "prefill_long", "kind": "prefill", "tokens": 3000, "outputs": "last"},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the listed ones' ranges."""
    kind = rng.choice(("apply", "apply", "sweep", "project", "project", "project", "lookup", "pack", "turn", "steps",
                       "prefill", "prefill"))
    bits = rng.choice((4, 4, 4, 2, 5))
    if kind == "apply":
        return {"kind": kind, "rows": _log(rng, 1, 512), "k": _log(rng, 128, 4096), "n": _log(rng, 64, 8192), "bits": bits}
    if kind == "sweep":
        return {"kind": kind, "count": _log(rng, 4, 32), "k": _log(rng, 256, 4096), "n": _log(rng, 512, 8192), "bits": bits}
    if kind == "project":
        rows, k = _log(rng, 2, 4096), 16 * _log(rng, 16, 256)
        n = _log(rng, 128, max(256, min(8192, 4096 * 768 * 8192 // (rows * k))))
        return {"kind": kind, "rows": rows, "k": k, "n": n, "bits": bits}
    if kind == "lookup":
        return {"kind": kind, "vocab": _log(rng, 1024, 32768), "k": _log(rng, 256, 2048), "ids": _log(rng, 1, 2048),
                "candidates": _log(rng, 1, 1000)}
    if kind == "pack":
        return {"kind": kind, "n": _log(rng, 64, 8192), "k": _log(rng, 128, 1024)}
    if kind == "turn":
        span = rng.random() < 0.5
        return {"kind": kind, "prompt": _log(rng, 5, 200), "fill": _log(rng, 8, 600) if span else 0,
                "ring": rng.randrange(64, 513) if span else 0, "steps": rng.randrange(1, 33)}
    if kind == "steps":
        return {"kind": kind, "context": _log(rng, 200, 2900), "steps": rng.randrange(1, 9)}
    outputs = rng.choice(("last", "last", "all"))
    return {"kind": kind, "tokens": _log(rng, 2, 3000 if outputs == "last" else 1000), "outputs": outputs}


# ------------------------------------------------------------------ inputs
# The code tables of the CQ format: the codebooks' centroids (over sqrt(128))
# and the int8 codebooks the products use, with their scales.
_C4 = ("-0x1.5ae0f408928fbp+1", "-0x1.05b0b8a516d54p+1", "-0x1.9841ff0758fc8p+0", "-0x1.3bbbebadac679p+0",
       "-0x1.d82c6dd21f59ep-1", "-0x1.47717151708b5p-1", "-0x1.7d9b9e4b565fap-2", "-0x1.d4ca474b8559bp-4",
       "0x1.2683e9154fce2p-3", "0x1.9daf49368793ap-2", "0x1.586b43e57d29dp-1", "0x1.ec3d50cbc3b33p-1",
       "0x1.4688db93b85f1p+0", "0x1.a3164906b428fp+0", "0x1.0ace7bbde2442p+1", "0x1.5ed98d06f2a4ap+1")
_C2 = ("-0x1.81b52e4028034p+0", "-0x1.ce467275b97c2p-2", "0x1.cfd177c54d348p-2", "0x1.828af1c856640p+0")
_TERNARY = 1.2240064


def _centroids(bits):
    """The f32 values by stored code (a ternary record's code 3 is its first level)."""
    if bits == 5:
        c = [0.0, _TERNARY, 0.0, -_TERNARY]
    else:
        c = [float.fromhex(v) for v in (_C4 if bits == 4 else _C2)]
    return (np.array(c) / math.sqrt(128.0)).astype(np.float32)


def _int8_codebook(bits):
    c = _centroids(bits).astype(np.float64)
    scale = np.abs(c).max() / 127.0
    v = c / scale
    return np.sign(v) * np.floor(np.abs(v) + 0.5), scale


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1_000_003 + 17)
    return g


def _codes(g, n, k, bits):
    """Codes [n][groups * 128] of Gaussian weights and their f16 group norms, on the device."""
    groups = (k + GROUP - 1) // GROUP
    x = torch.randn(n, groups * GROUP, generator=g, device="cuda") / math.sqrt(128.0)
    cb = torch.from_numpy(_centroids(bits)).cuda()
    if bits == 5:  # levels -t, 0, t as codes 3, 0, 1
        codes = torch.where(x < cb[3] / 2, 3, torch.where(x > cb[1] / 2, 1, 0)).to(torch.uint8)
    else:
        codes = torch.bucketize(x, (cb[1:] + cb[:-1]) / 2).to(torch.uint8)
    norms = (0.02 * math.sqrt(128.0) * (1 + 0.06 * torch.randn(n, groups, generator=g, device="cuda"))).half()
    return codes, norms


def _packed(codes, bits):
    """Least significant first, two codes to a byte (4-bit) or four."""
    per = 2 if bits == 4 else 4
    c = codes.view(codes.shape[0], -1, per)
    out = torch.zeros_like(c[..., 0])
    for i in range(per):
        out |= c[..., i] << (i * (8 // per))
    return out.cpu().numpy()


def _matrix(g, n, k, bits):
    codes, norms = _codes(g, n, k, bits)
    return nh.QMat.from_cq(_packed(codes, bits), norms.cpu().numpy().view(np.uint16), n, k, bits)


def _parts(n):
    """A fused projection's parts: q | k | v | gate for a Needle-3 layer, else a half and the rest."""
    return QKVG if n == sum(QKVG) else (n - n // 2, n // 2)


@functools.lru_cache(maxsize=1)
def _model():
    """Random weights of the published Needle-3 architecture, loaded once per program."""
    return nh.Model.from_archive(archive.random_needle3(nh, archive.Needle3(vocab=VOCAB), seed=0))


def _tokens(seed, n):
    return np.random.default_rng(seed).integers(0, VOCAB, n).astype(np.uint32)


def prepare(case, seed):
    nh.init(0)
    kind = case["kind"]
    if kind in ("turn", "steps", "prefill"):
        model = _model()
    if kind == "turn":
        total = case["prompt"] + case["fill"] + case["steps"]
        return {"case": case, "session": model.session(total), "toks": _tokens(seed, case["prompt"] + case["fill"])}
    if kind == "steps":
        toks = _tokens(seed, case["context"] + case["steps"])
        sess = model.session(case["context"] + case["steps"])
        sess.prefill(toks[:case["context"]], nh.OUT_NONE)
        return {"case": case, "session": sess, "toks": toks}
    if kind == "prefill":
        return {"case": case, "session": model.session(case["tokens"]), "toks": _tokens(seed, case["tokens"])}
    if kind == "pack":
        rng = np.random.default_rng(seed)
        return {"case": case, "w": rng.standard_normal((case["n"], case["k"]), dtype=np.float32) * np.float32(0.02)}
    g = _generator(seed)
    if kind == "apply":
        lin = nh.QLinear([_matrix(g, n, case["k"], case["bits"]) for n in _parts(case["n"])])
        return {"case": case, "lin": lin, "x": torch.randn(case["rows"], case["k"], generator=g, device="cuda")}
    if kind == "sweep":
        mats = [_matrix(g, case["n"], case["k"], case["bits"]) for _ in range(case["count"])]
        x = torch.randn(1, case["k"], generator=g, device="cuda")
        a = nh.QAct.new(x, 1, case["k"], mats[0].act_bits())
        ys = torch.empty(case["count"], 1, case["n"], device="cuda")

        def sweep():
            for m, y in zip(mats, ys):
                m.matmul_into(a, y, case["n"], 0)

        sweep()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            sweep()
        return {"case": case, "mats": mats, "a": a, "ys": ys, "graph": graph}
    if kind == "project":
        mat = _matrix(g, case["n"], case["k"], case["bits"])
        x = torch.randn(case["rows"], case["k"], generator=g, device="cuda") * 3
        scale = (0.1 * torch.randn(case["k"], generator=g, device="cuda")).half()
        return {"case": case, "mat": mat, "x": x, "scale": scale,
                "a": nh.QAct.empty_rows(case["rows"], case["k"], mat.act_bits())}
    if kind == "lookup":
        mat = _matrix(g, case["vocab"], case["k"], 4)
        h = torch.randn(1, case["k"], generator=g, device="cuda")
        ids = torch.randint(0, case["vocab"], (case["ids"],), generator=g, device="cuda").int()
        cand = torch.randperm(case["vocab"], generator=g, device="cuda")[:case["candidates"]].int()
        return {"case": case, "mat": mat, "h": h, "ids": ids, "cand": cand,
                "a": nh.QAct.empty_rows(1, case["k"], 4)}
    raise ValueError(kind)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "apply":
        return state["lin"].apply(state["x"], case["rows"])
    if kind == "sweep":
        state["graph"].replay()
        return state["ys"]
    if kind == "project":
        state["a"].prep(state["x"], case["rows"], state["scale"])
        return state["mat"].matmul(state["a"])
    if kind == "lookup":
        rows = state["mat"].rows(state["ids"])
        state["a"].prep(state["h"], 1)
        return rows, nh.head_logits_sparse(state["mat"], state["a"], state["cand"], case["vocab"])
    if kind == "pack":
        return nh.QMat.from_f32(state["w"], case["n"], case["k"]).download()
    sess, toks = state["session"], state["toks"]
    if kind == "turn":
        sess.reset()
        if case["ring"]:
            sess.set_attend(case["prompt"], case["ring"])
            sess.prefill(toks[:case["prompt"]], nh.OUT_NONE)
            sess.prefill(toks[case["prompt"]:])
        else:
            sess.forward(toks)
        return sess.generate_greedy(case["steps"])
    if kind == "steps":
        if len(sess) > case["context"]:
            sess.rollback(len(sess) - case["context"])
        return [sess.forward(toks[i:i + 1]) for i in range(case["context"], case["context"] + case["steps"])]
    sess.reset()
    return sess.forward(toks) if case["outputs"] == "last" else sess.forward(toks, nh.OUT_ALL_LOGITS)


# ------------------------------------------------------------------- work
def _cq_bytes(n, k, bits):
    groups = (k + GROUP - 1) // GROUP
    return n * groups * (GROUP * (4 if bits == 4 else 2) // 8 + 2)


def _forward_work(first, last, heads):
    """Positions first .. last - 1 of the default Needle-3 through its 20 layers (4 of them global, the rest
    with a window of 1,024), `heads` rows of logits: the weights once, the keys and values that the positions
    see once, the new ones written."""
    n, layers, d = last - first, 20, 768
    per_layer = 1568 * d + d * d + 24 * 4 * d  # q|k|v|gate, out, the mHC rows
    engram = 5 * 2 * d * d
    mlp = 3 * 1024 * 32 * 2  # the six Kronecker passes' multiply-adds
    keys_global = sum(range(first + 1, last + 1))
    keys_window = sum(min(i, 1024) for i in range(first + 1, last + 1))
    attend = 2 * 12 * (48 + 64) * (4 * keys_global + 16 * keys_window)
    flops = 2 * n * (layers * (per_layer + mlp) + engram) + attend + 2 * heads * VOCAB * d
    cache = 2 * (48 + 4 + 64)
    seen = 4 * last + 16 * min(last, 1024 + n)
    weights = _cq_bytes(layers * 2336 + 5 * 2 * d + (VOCAB if heads else 0), d, 4) + layers * 24 * 4 * d
    return {"bytes": weights + cache * seen + n * 4 * d + heads * VOCAB * 4, "flops": flops}


def work(case):
    kind = case["kind"]
    if kind in ("apply", "project"):
        m, k, n = case["rows"], case["k"], case["n"]
        return {"bytes": _cq_bytes(n, k, case["bits"]) + 4 * m * (k + n), "flops": 2 * m * n * k}
    if kind == "sweep":
        k, n = case["k"], case["n"]
        return {"bytes": case["count"] * (_cq_bytes(n, k, case["bits"]) + 4 * n) + k, "flops": 2 * case["count"] * n * k}
    if kind == "lookup":
        k, ids, cand = case["k"], case["ids"], case["candidates"]
        return {"bytes": _cq_bytes(ids + cand, k, 4) + 4 * (ids * k + k + case["vocab"] + ids + cand),
                "flops": ids * k * 9 + 2 * cand * k}
    if kind == "pack":
        n, k = case["n"], case["k"]
        return {"bytes": 4 * n * k + _cq_bytes(n, k, 4), "flops": n * k * 30}
    if kind == "turn":
        p = case["prompt"] + case["fill"]
        seen = [_forward_work(0, p, 1)]
        for i in range(p, p + case["steps"]):
            seen.append(_forward_work(i, i + 1, 1))
            if case["ring"]:  # a span's query sees its sink and its ring
                keys = min(i + 1, case["prompt"] + case["ring"])
                seen[-1] = _forward_work(keys - 1, keys, 1)
        return {f: sum(s[f] for s in seen) for f in ("bytes", "flops")}
    if kind == "steps":
        seen = [_forward_work(i, i + 1, 1) for i in range(case["context"], case["context"] + case["steps"])]
        return {f: sum(s[f] for s in seen) for f in ("bytes", "flops")}
    return _forward_work(0, case["tokens"], 1 if case["outputs"] == "last" else case["tokens"])


def tolerance(case):
    """Results are fixed to the bit: the integer sums are exact, and the order and rounding of every float
    operation around them is part of the format's arithmetic (two correct programs give the same bytes)."""
    return "exact"


# ------------------------------------------------------------------ 64 bits
def _rotate(x):
    """The normalised 128-point Hadamard rotation of every group of the last axis."""
    h = torch.ones(1, 1, dtype=torch.float64, device=x.device)
    while h.shape[0] < GROUP:
        h = torch.cat((torch.cat((h, h), 1), torch.cat((h, -h), 1)), 0)
    return (x.view(*x.shape[:-1], -1, GROUP) @ (h / math.sqrt(GROUP))).view(x.shape)


def _pad(x):
    return torch.nn.functional.pad(x, (0, -x.shape[-1] % GROUP))


def _a8(x):
    """Rows [m][k] as rotated int8 codes [m][groups][128] and group scales, in 64 bits."""
    v = _rotate(_pad(x.double()))
    v = v.view(v.shape[0], -1, GROUP)
    s = v.abs().amax(-1, keepdim=True) / 127.0
    s = torch.where(s > 0, s, torch.ones_like(s))
    q = v / s
    return torch.sign(q) * torch.floor(q.abs() + 0.5), s


def _product(x, codes, norms, bits):
    q, s = _a8(x)
    cb, scale = _int8_codebook(bits)
    w = torch.from_numpy(cb).cuda()[codes.long()].view(codes.shape[0], -1, GROUP)
    w = w * (norms.double() * scale)[..., None]
    return (q * s).reshape(x.shape[0], -1) @ w.reshape(codes.shape[0], -1).T


def _pack64(w):
    v = _rotate(_pad(torch.from_numpy(w).double().cuda()))
    v = v.view(w.shape[0], -1, GROUP)
    norm = v.square().sum(-1, keepdim=True).sqrt()
    cb = torch.from_numpy(_centroids(4).astype(np.float64)).cuda()
    codes = torch.bucketize((v / norm.clamp_min(1e-12)).contiguous(), (cb[1:] + cb[:-1]) / 2).to(torch.uint8)
    return _packed(codes.view(w.shape[0], -1), 4), norm[..., 0].half().cpu().numpy().view(np.uint16)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("turn", "steps", "prefill"):
        # Twenty layers that each round their activations to int8: a 64-bit
        # evaluation rounds other activations up than these do, and its
        # logits are those of another rounding, not a value they approach.
        return None
    if kind == "pack":
        return _pack64(prepare(case, seed)["w"])
    g = _generator(seed)
    k = case["k"]
    if kind == "apply":
        mats = [_codes(g, n, k, case["bits"]) for n in _parts(case["n"])]
        x = torch.randn(case["rows"], k, generator=g, device="cuda")
        return torch.cat([_product(x, c, n, case["bits"]) for c, n in mats], 1)
    if kind == "sweep":
        mats = [_codes(g, case["n"], k, case["bits"]) for _ in range(case["count"])]
        x = torch.randn(1, k, generator=g, device="cuda")
        return torch.stack([_product(x, c, n, case["bits"]) for c, n in mats])
    if kind == "project":
        codes, norms = _codes(g, case["n"], k, case["bits"])
        x = torch.randn(case["rows"], k, generator=g, device="cuda") * 3
        scale = (0.1 * torch.randn(k, generator=g, device="cuda")).half()
        x = x.double()
        x = x / (x.square().mean(-1, keepdim=True) + 1e-6).sqrt() * (1 + scale.double())
        return _product(x, codes, norms, case["bits"])
    codes, norms = _codes(g, case["vocab"], k, 4)
    h = torch.randn(1, k, generator=g, device="cuda")
    ids = torch.randint(0, case["vocab"], (case["ids"],), generator=g, device="cuda")
    cand = torch.randperm(case["vocab"], generator=g, device="cuda")[:case["candidates"]]
    cb = torch.from_numpy(_centroids(4).astype(np.float64)).cuda()
    w = cb[codes[ids].long()].view(ids.numel(), -1, GROUP) * norms[ids].double()[..., None]
    rows = _rotate(w.reshape(ids.numel(), -1))[:, :k]
    logits = torch.full((case["vocab"],), float(np.float32(-1e30)), dtype=torch.float64, device="cuda")
    logits[cand] = _product(h, codes[cand], norms[cand], 4)[0]
    return rows, logits
