"""Workloads that stand for what a user of this package has it do.

Each case is a dict of plain values; its "kind" names the entry points it
goes through:

  linear    srq_linear_enqueue: one weight matrix (Q8, Q4 or F32) times n
            activation rows on the device -- one row while decoding, 5..64 in a
            continuous-batching step, up to 1024 in a prefill chunk
  pack      srq_pack: a bf16 / f16 / f32 matrix to Q8 or Q4 (the load path)
  prompt    Model.step over the chunks of one prompt: prefill through whole
            decoder layers and the head, host logits of the last position
  generate  Model.generate_greedy, then one more step for the logits: prefill,
            graph-replayed decode and the device argmax
  serve     TickPlanner's continuous-batching ticks over many sessions, each
            a Model.step followed by sample on the device-resident logits
  sample    sample: token sampling over the logits rows of a step

Models are a few layers of the shapes in sr_go_tranformer_amd/synthetic.py
(SmolLM2-135M whole), since a layer's work does not depend on how many follow.

Weights are made as code * scale with a scale of few significant bits and a
full-range code in every 64-column block, so that packing them gives back
exactly these codes and scales: the dense values are what every format
computes with, and the 64-bit reference needs no packer of its own.
"""
import ctypes as C
import math

import numpy as np
import torch

import sr_go_tranformer_amd as srq
from sr_go_tranformer_amd import synthetic
from sr_go_tranformer_amd.schedule import TickPlanner

FMT = {"f32": srq.F32, "q8": srq.Q8, "q4": srq.Q4}
SRC = {"f32": srq.SRC_F32, "bf16": srq.SRC_BF16, "f16": srq.SRC_F16}
TORCH_SRC = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
LEVELS = {"q8": 127, "q4": 7}
BLOCK, PAGE = 64, 32
DEV = "cuda:0"

_executor = None


def executor():
    """The program's one executor (one stream, one workspace)."""
    global _executor
    if _executor is None:
        _executor = srq.Executor(0)
    return _executor


# ------------------------------------------------------------------- cases


def listed():
    return [
        # The smallest call: SmolLM2-135M's down projection for one token.
        # Latency: the launch, one round of loads, the reduction.
        dict(name="linear-q8-576x1536-n1", kind="linear", fmt="q8", rows=576, cols=1536, n=1),
        # Mistral-7B's fused gate/up matrix for one token: the matrix that
        # dominates Q8 decode, bound by HBM.
        dict(name="linear-q8-28672x4096-n1", kind="linear", fmt="q8", rows=28672, cols=4096, n=1),
        # Llama-3.2-3B's gate/up for the rows of one continuous-batching step.
        dict(name="linear-q8-16384x3072-n32", kind="linear", fmt="q8", rows=16384, cols=3072, n=32),
        # Mistral-7B's gate/up for a prefill chunk of 256 tokens, Q4.
        dict(name="linear-q4-28672x4096-n256", kind="linear", fmt="q4", rows=28672, cols=4096, n=256),
        # Mistral-7B's down projection for the largest chunk a step takes,
        # with a ragged last tile.
        dict(name="linear-q8-4096x14336-n1000", kind="linear", fmt="q8", rows=4096, cols=14336, n=1000),
        # SmolLM2-135M's gate/up kept in F32, a ragged prompt.
        dict(name="linear-f32-3072x576-n129", kind="linear", fmt="f32", rows=3072, cols=576, n=129),
        # One checkpoint matrix (Mistral-7B up projection, bf16) packed at load.
        dict(name="pack-q8-14336x4096-bf16", kind="pack", fmt="q8", rows=14336, cols=4096, src="bf16"),
        # Prefill of a 2048-token prompt in 256-token chunks, two
        # Mistral-7B-width layers with Q4 matrices, Q8 embedding and head.
        dict(name="prompt-7b-q4mixed-2048", kind="prompt", shape="mistral-7b", layers=2, fmt="q4-mixed", prompt=2048,
             chunk=256),
        # SmolLM2-135M whole, Q8: 32-token prompt, 64 greedy tokens.
        dict(name="generate-smollm-q8", kind="generate", shape="smollm2-135m", layers=30, fmt="q8", prompt=32,
             count=64, chunk=16),
        # Four Mistral-7B-width layers, Q4 matrices: 128-token prompt, 32
        # greedy tokens.
        dict(name="generate-7b-q4mixed", kind="generate", shape="mistral-7b", layers=4, fmt="q4-mixed", prompt=128,
             count=32, chunk=128),
        # Continuous batching over four Llama-3.2-3B-width layers, Q8, at the
        # engine's scheduling and sampling defaults.
        dict(name="serve-3b-q8-32", kind="serve", shape="llama3.2-3b", layers=4, fmt="q8", sessions=32, prompt=96,
             count=12, temperature=0.8, top_k=40, top_p=0.95, penalty=1.1),
        # Sampling of one 32-session step over a 128256-id vocabulary, no
        # top-k cut.
        dict(name="sample-32x128256", kind="sample", rows=32, vocab=128256, temperature=0.8, top_k=0, top_p=0.9,
             penalty=1.0, history=0),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case: sizes over the ranges above (log-uniform), odd widths,
    heights and row counts among them."""
    kind = rng.choice(["linear"] * 5 + ["pack", "prompt", "generate", "serve", "sample"])
    if kind == "linear":
        fmt = rng.choice(["q8", "q8", "q4", "q4", "f32"])
        while True:
            n = _log(rng, 1, 1024)
            rows = _log(rng, 64, 32768)
            cols = _log(rng, 64, 14336)
            if rng.random() < 0.85:
                cols = max(64, cols // 64 * 64)
            if rng.random() < 0.6:
                rows = max(64, rows // 32 * 32)
            # widths that are no multiple of 32 take the row-by-row path; no
            # model has them with long chunks
            if cols % 32 and n > 16:
                continue
            if rows * cols <= 28672 * 4096 and n * rows * cols <= (20e9 if fmt != "f32" else 4e9):
                break
        return dict(kind=kind, fmt=fmt, rows=rows, cols=cols, n=n)
    if kind == "pack":
        return dict(kind=kind, fmt=rng.choice(["q8", "q4"]), rows=_log(rng, 64, 14336), cols=_log(rng, 64, 8192),
                    src=rng.choice(["bf16", "f16", "f32"]))
    if kind == "prompt":
        return dict(kind=kind, shape=rng.choice(["smollm2-135m", "llama3.2-1b", "mistral-7b"]),
                    layers=rng.choice([1, 2]), fmt=rng.choice(["q8", "q4", "q4-mixed"]), prompt=_log(rng, 24, 2048),
                    chunk=rng.choice([16, 64, 256, 500, 1024]))
    if kind == "generate":
        return dict(kind=kind, shape=rng.choice(["smollm2-135m", "llama3.2-1b", "mistral-7b"]),
                    layers=rng.choice([1, 2, 4]), fmt=rng.choice(["q8", "q4-mixed"]), prompt=_log(rng, 8, 1500),
                    count=rng.randint(8, 40), chunk=rng.choice([16, 128, 512]))
    if kind == "serve":
        return dict(kind=kind, shape=rng.choice(["smollm2-135m", "llama3.2-1b", "llama3.2-3b"]),
                    layers=rng.choice([1, 2]), fmt=rng.choice(["q8", "q4-mixed"]), sessions=_log(rng, 2, 32),
                    prompt=_log(rng, 16, 96), count=rng.randint(4, 12), temperature=0.8, top_k=40, top_p=0.95,
                    penalty=1.1)
    return dict(kind=kind, rows=_log(rng, 1, 48), vocab=_log(rng, 1000, 128256),
                temperature=rng.choice([0.6, 0.8, 1.0]), top_k=rng.choice([0, 0, 40]),
                top_p=rng.choice([0.9, 0.95, 1.0]), penalty=rng.choice([1.0, 1.1]), history=_log(rng, 1, 200))


# ------------------------------------------------------------------ inputs


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) & 0x7FFFFFFFFFFF)
    return g


def _dense(g, rows, cols, fmt, std=0.02):
    """N(0, std) weights whose packed form is exact (see above)."""
    w = torch.randn(rows, cols, generator=g, device=DEV) * std
    if fmt == "f32":
        return w
    levels = LEVELS[fmt]
    pad = -cols % BLOCK
    b = torch.nn.functional.pad(w, (0, pad)).view(rows, -1, BLOCK)
    top, at = b.abs().max(dim=2, keepdim=True)
    scale = (top / levels).bfloat16().float().clamp_min(2.0**-60)
    code = (b / scale).round_().clamp_(-levels, levels)
    full = torch.where(b.gather(2, at) < 0, -float(levels), float(levels))
    code.scatter_(2, at, full)
    return (code * scale).view(rows, -1)[:, :cols].contiguous()


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _formats(fmt):
    """(layer matrices, embedding and head)"""
    return ("q4", "q8") if fmt == "q4-mixed" else (fmt, fmt)


def _tensors(case, seed):
    """(kind, layer, name, dense tensor) of a model in the order they are loaded."""
    s = synthetic.SHAPES[case["shape"]]
    d, H, V = s["dim"], s["hidden"], s["vocab"]
    kd = d // s["heads"] * s["kv_heads"]
    fl, fe = _formats(case["fmt"])
    g = _gen(seed)

    def norm():
        return 1.0 + 0.1 * torch.randn(d, generator=g, device=DEV)

    yield srq.T_EMBED, 0, "embed", _dense(g, V, d, fe)
    for l in range(case["layers"]):
        yield srq.T_ATTN_NORM, l, "n1", norm()
        for kind, name, r, c in ((srq.T_Q, "q", d, d), (srq.T_K, "k", kd, d), (srq.T_V, "v", kd, d), (srq.T_O, "o", d, d)):
            yield kind, l, name, _dense(g, r, c, fl)
        yield srq.T_FFN_NORM, l, "n2", norm()
        for kind, name, r, c in ((srq.T_GATE, "gate", H, d), (srq.T_UP, "up", H, d), (srq.T_DOWN, "down", d, H)):
            yield kind, l, name, _dense(g, r, c, fl)
    yield srq.T_FINAL_NORM, 0, "norm", norm()
    if not s["tied"]:
        yield srq.T_OUTPUT, 0, "head", _dense(g, V, d, fe)


def _context(case):
    return (case["prompt"] + case.get("count", 0) + 2 + PAGE - 1) // PAGE * PAGE


def _model(case, seed):
    s = synthetic.SHAPES[case["shape"]]
    cfg = srq.make_config(s["vocab"], s["dim"], case["layers"], s["heads"], s["kv_heads"], s["hidden"], _context(case),
                          s["rope_theta"], 1e-5, s["tied"])
    m = srq.Model(executor(), cfg, case["fmt"])
    for kind, layer, _, t in _tensors(case, seed):
        torch.cuda.synchronize()  # the executor's stream does not wait for torch's
        m.load_device(kind, layer, t.data_ptr())
    return m


def _tokens(rng, count, vocab):
    return [int(t) for t in rng.integers(0, vocab, count)]


def _requests(case, seed):
    """Prompts of 1/6 to all of case["prompt"] tokens and their continuations."""
    rng = np.random.default_rng(seed)
    V = synthetic.SHAPES[case["shape"]]["vocab"]
    prompts = [_tokens(rng, int(rng.integers(max(1, case["prompt"] // 6), case["prompt"] + 1)), V)
               for _ in range(case["sessions"])]
    return prompts, [_tokens(rng, case["count"], V) for _ in prompts]


def prepare(case, seed):
    k = case["kind"]
    ex = executor()
    st = {"case": case, "kind": k, "ex": ex}
    if k == "linear":
        g = _gen(seed)
        w = _dense(g, case["rows"], case["cols"], case["fmt"])
        st["x"] = torch.randn(case["n"], case["cols"], generator=g, device=DEV)
        st["y"] = torch.zeros(case["n"], case["rows"], device=DEV)
        torch.cuda.synchronize()
        h = C.c_void_p()
        srq.check(srq.lib().srq_weight_create(ex.h, FMT[case["fmt"]], case["rows"], case["cols"], _ptr(w), srq.SRC_F32,
                                              C.byref(h)))
        st["w"] = srq.Weight(h)
    elif k == "pack":
        st["src"] = _pack_source(case, seed)
        vb, sb = srq.packed_bytes(FMT[case["fmt"]], case["rows"], case["cols"])
        st["values"] = torch.zeros(vb, dtype=torch.uint8, device=DEV)
        st["scales"] = torch.zeros(sb // 4, device=DEV)
    elif k == "sample":
        rng = np.random.default_rng(seed)
        st["logits"] = 2.5 * torch.randn(case["rows"], case["vocab"], generator=_gen(seed), device=DEV)
        st["rng"] = rng.integers(0, 1 << 63, case["rows"]).astype(np.uint64)
        st["histories"] = None
        if case["penalty"] != 1.0:
            st["histories"] = [_tokens(rng, case["history"], case["vocab"]) for _ in range(case["rows"])]
        st["params"] = srq.Sampling(case["temperature"], case["top_k"], case["top_p"], case["penalty"])
    else:
        st["m"] = _model(case, seed)
        pages = _context(case) // PAGE
        st["pages"] = pages
        st["pool"] = st["m"].pool(pages * case.get("sessions", 1))
        if k == "serve":
            st["prompts"], st["forced"] = _requests(case, seed)
            st["rng"] = np.random.default_rng(seed + 1).integers(0, 1 << 63, case["sessions"]).astype(np.uint64)
            st["params"] = srq.Sampling(case["temperature"], case["top_k"], case["top_p"], case["penalty"])
            st["logits"] = torch.zeros(case["sessions"], st["m"].config.vocab, device=DEV)
        else:
            st["ids"] = np.array(_tokens(np.random.default_rng(seed), case["prompt"], st["m"].config.vocab), np.int32)
    torch.cuda.synchronize()
    return st


def _pack_source(case, seed):
    w = torch.randn(case["rows"], case["cols"], generator=_gen(seed), device=DEV) * 0.02
    return w.to(TORCH_SRC[case["src"]])


# --------------------------------------------------------------------- run


def run(st):
    return {"linear": _run_linear, "pack": _run_pack, "sample": _run_sample, "prompt": _run_prompt,
            "generate": _run_generate, "serve": _run_serve}[st["kind"]](st)


def _run_linear(st):
    srq.check(srq.lib().srq_linear_enqueue(st["ex"].h, _ptr(st["y"]), _ptr(st["x"]), st["w"].h, st["case"]["n"]))
    return st["y"]


def _run_pack(st):
    c = st["case"]
    srq.check(srq.lib().srq_pack(st["ex"].h, FMT[c["fmt"]], c["rows"], c["cols"], _ptr(st["src"]), SRC[c["src"]],
                                 _ptr(st["values"]), _ptr(st["scales"])))
    return {"values": st["values"], "scales": st["scales"]}


def _run_sample(st):
    rng = st["rng"].copy()
    c = st["case"]
    ids = srq.sample(st["ex"], _ptr(st["logits"]), c["rows"], c["vocab"], st["params"], rng, histories=st["histories"])
    return {"ids": ids, "rng": rng.view(np.int64)}


def _run_prompt(st):
    c, m, ids = st["case"], st["m"], st["ids"]
    cache = st["pool"].cache(st["pages"])
    for a in range(0, len(ids), c["chunk"]):
        last = a + c["chunk"] >= len(ids)
        out = m.step([cache], [ids[a:a + c["chunk"]]], want=[last], host=last)
    cache.close()
    return out


def _run_generate(st):
    c, m = st["case"], st["m"]
    cache = st["pool"].cache(st["pages"])
    toks = m.generate_greedy(cache, st["ids"], c["count"], chunk=c["chunk"])
    out = m.step([cache], [[toks[-1]]])
    cache.close()
    return {"tokens": np.array(toks, np.int64), "logits": out}


def _run_serve(st):
    """The engine's ticks, every completed session sampled each tick.  The
    continuations that go back in are given, as when a logged session is
    replayed, so that one draw does not decide all that follows; a last
    step of every session leaves its logits."""
    c, m = st["case"], st["m"]
    vocab = m.config.vocab
    caches = [st["pool"].cache(st["pages"]) for _ in st["prompts"]]
    rng = st["rng"].copy()
    drawn = [[] for _ in caches]
    history = [list(p) for p in st["prompts"]]
    plan = TickPlanner(st["prompts"], c["count"])
    while not plan.done():
        sessions, chunks, want = plan.plan()
        dev = m.step([caches[i] for i in sessions], chunks, want=want, host=False)
        rows = [k for k, w in enumerate(want) if w]
        sampled = {}
        if rows:
            who = [sessions[k] for k in rows]
            state = rng[who]
            ids = srq.sample(st["ex"], dev, len(rows), vocab, st["params"], state, histories=[history[i] for i in who],
                             row_ids=rows)
            rng[who] = state
            for i, t in zip(who, ids):
                drawn[i].append(int(t))
                sampled[i] = st["forced"][i][len(drawn[i]) - 1]
                history[i].append(sampled[i])
        plan.commit(sampled)
    dev = m.step(caches, [[f[-1]] for f in st["forced"]], host=False)
    srq.check(srq.lib().srq_copy_d2d(st["ex"].h, _ptr(st["logits"]), dev, st["logits"].numel() * 4))
    for cache in caches:
        cache.close()
    return {"ids": np.array(drawn, np.int64), "logits": st["logits"]}


# -------------------------------------------------------------------- work


def _matrix_bytes(fmt, rows, cols):
    v, s = srq.packed_bytes(FMT[fmt], rows, cols) if fmt != "f32" else (rows * cols * 4, 0)
    return v + s


def _model_work(case, steps):
    """steps: per step (rows, context positions its rows attend to in all,
    logits rows).  Every step reads the layers' matrices once, and the head
    if it returns logits."""
    s = synthetic.SHAPES[case["shape"]]
    d, H, V = s["dim"], s["hidden"], s["vocab"]
    kd = d // s["heads"] * s["kv_heads"]
    fl, fe = _formats(case["fmt"])
    shapes = [(d + 2 * kd, d), (d, d), (2 * H, d), (d, H)]
    weights = case["layers"] * sum(_matrix_bytes(fl, r, c) for r, c in shapes)
    params = case["layers"] * sum(r * c for r, c in shapes)
    b = f = 0.0
    for n, attended, longest, heads in steps:
        b += weights + n * d * 4 + case["layers"] * (longest * 2 * kd * 4) + heads * V * 4
        f += 2.0 * n * params + case["layers"] * 4.0 * attended * d + 2.0 * heads * V * d
        if heads:
            b += _matrix_bytes(fe, V, d)
    return {"bytes": b, "flops": f}


def _chunk_steps(prompt, chunk, last_heads=1):
    out = []
    for a in range(0, prompt, chunk):
        e = min(prompt, a + chunk)
        out.append((e - a, sum(range(a + 1, e + 1)), e, last_heads if e == prompt else 0))
    return out


def work(case):
    k = case["kind"]
    if k == "linear":
        n, r, c = case["n"], case["rows"], case["cols"]
        return {"bytes": _matrix_bytes(case["fmt"], r, c) + 4.0 * n * (r + c), "flops": 2.0 * n * r * c}
    if k == "pack":
        r, c = case["rows"], case["cols"]
        return {"bytes": float(r * c * (4 if case["src"] == "f32" else 2) + _matrix_bytes(case["fmt"], r, c)),
                "flops": 0.0}
    if k == "sample":
        return {"bytes": 4.0 * case["rows"] * case["vocab"], "flops": 0.0}
    if k == "prompt":
        return _model_work(case, _chunk_steps(case["prompt"], case["chunk"]))
    if k == "generate":
        p = case["prompt"]
        return _model_work(case, _chunk_steps(p, case["chunk"]) +
                           [(1, p + i + 1, p + i + 1, 1) for i in range(case["count"])])
    # serve: every tick's rows are known from the prompts' lengths; a middling
    # seed stands for all
    prompts, forced = _requests(case, 0)
    plan, pos, steps = TickPlanner(prompts, case["count"]), [0] * len(prompts), []
    while not plan.done():
        sessions, chunks, want = plan.plan()
        n = attended = longest = 0
        for i, ch in zip(sessions, chunks):
            attended += sum(range(pos[i] + 1, pos[i] + len(ch) + 1))
            pos[i] += len(ch)
            n += len(ch)
            longest += pos[i]
        steps.append((n, attended, longest, sum(want)))
        plan.commit({i: forced[i][0] for i, w in zip(sessions, want) if w})
    return _model_work(case, steps)


# --------------------------------------------------------------- tolerance


def tolerance(case):
    """Everything is accumulated in 32 bits from operands held exactly: about
    four times the distance from 64 bits that was measured (1e-7 for one Q8 /
    Q4 product, 3e-7 for F32 weights, 2e-6 for logits through two layers of
    2048 positions).  Packing and sampling give whole numbers; a few of a
    served run's draws may fall between two orders of a near tie."""
    k = case["kind"]
    if k == "linear":
        return {"rel": 1.5e-6 if case["fmt"] == "f32" else 6e-7, "max": 2e-5}
    if k == "pack":
        return "exact"
    if k == "sample":
        return "exact"
    return {"rel": 1e-5, "max": 2e-4, "differ": 0.01}


# ------------------------------------------------------------------- exact


def exact(case, seed):
    k = case["kind"]
    if k == "linear":
        g = _gen(seed)
        w = _dense(g, case["rows"], case["cols"], case["fmt"])
        x = torch.randn(case["n"], case["cols"], generator=g, device=DEV)
        return x.double() @ w.double().T
    if k == "pack":
        w = _pack_source(case, seed).double()
        pad = -case["cols"] % BLOCK
        top = torch.nn.functional.pad(w, (0, pad)).view(case["rows"], -1, BLOCK).abs().amax(dim=2)
        return {"values": None, "scales": (top / LEVELS[case["fmt"]]).reshape(-1)}
    if k == "sample":
        return None
    ref = _Reference(case, seed)
    V = synthetic.SHAPES[case["shape"]]["vocab"]
    if k == "serve":
        prompts, forced = _requests(case, seed)
        return {"ids": None, "logits": torch.cat([ref.logits(ref.start(), p + f) for p, f in zip(prompts, forced)])}
    kv = ref.start()
    out = ref.logits(kv, _tokens(np.random.default_rng(seed), case["prompt"], V))
    if k == "prompt":
        return out
    for _ in range(case["count"]):
        out = ref.logits(kv, [int(out.argmax())])
    return {"tokens": None, "logits": out}


class _Reference:
    """The decoder in 64 bits, plain torch."""

    def __init__(self, case, seed):
        self.s = synthetic.SHAPES[case["shape"]]
        self.layers = case["layers"]
        self.t = {(name, l): t for _, l, name, t in _tensors(case, seed)}
        hd = self.s["dim"] // self.s["heads"]
        # inverse frequencies and angles are 32-bit by definition
        e = np.arange(0, hd, 2).astype(np.float32) / np.float32(hd)
        inv = np.float32(1) / np.power(self.s["rope_theta"], e.astype(np.float64)).astype(np.float32)
        ang = (np.arange(_context(case), dtype=np.float32)[:, None] * inv[None, :]).astype(np.float32)
        ang = torch.from_numpy(ang.astype(np.float64)).to(DEV)
        self.cos, self.sin = ang.cos(), ang.sin()

    def start(self):
        return {"pos": 0, "k": [None] * self.layers, "v": [None] * self.layers}

    def mul(self, x, name, l):
        return x @ self.t[name, l].double().T

    @staticmethod
    def norm(x, w):
        return x * torch.rsqrt(x.square().mean(dim=1, keepdim=True) + 1e-5) * w.double()

    def rope(self, x, pos, n):
        h = x.shape[-1] // 2
        c, s = self.cos[pos:pos + n, None], self.sin[pos:pos + n, None]
        a, z = x[..., :h], x[..., h:]
        return torch.cat([a * c - z * s, a * s + z * c], dim=-1)

    def logits(self, kv, tokens):
        s, n, pos = self.s, len(tokens), kv["pos"]
        hq, hk, hd = s["heads"], s["kv_heads"], s["dim"] // s["heads"]
        x = self.t["embed", 0][torch.tensor(tokens, device=DEV)].double()
        for l in range(self.layers):
            h = self.norm(x, self.t["n1", l])
            q = self.rope(self.mul(h, "q", l).view(n, hq, hd), pos, n)
            k = self.rope(self.mul(h, "k", l).view(n, hk, hd), pos, n)
            v = self.mul(h, "v", l).view(n, hk, hd)
            if pos:
                k, v = torch.cat([kv["k"][l], k]), torch.cat([kv["v"][l], v])
            kv["k"][l], kv["v"][l] = k, v
            past = torch.arange(pos + n, device=DEV)[None, :] <= torch.arange(pos, pos + n, device=DEV)[:, None]
            out = torch.empty(n, hq, hd, dtype=torch.float64, device=DEV)
            for i in range(hq):
                j = i * hk // hq
                w = (q[:, i] @ k[:, j].T) / math.sqrt(hd)
                out[:, i] = torch.softmax(w.masked_fill(~past, -math.inf), dim=1) @ v[:, j]
            x = x + self.mul(out.view(n, -1), "o", l)
            h = self.norm(x, self.t["n2", l])
            x = x + self.mul(torch.nn.functional.silu(self.mul(h, "gate", l)) * self.mul(h, "up", l), "down", l)
        kv["pos"] = pos + n
        last = self.norm(x[-1:], self.t["norm", 0])
        return self.mul(last, "embed" if s["tied"] else "head", 0)
