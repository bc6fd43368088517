"""Workloads that the speed of this library is judged by: the calls a program makes that runs one of the
supported language models on it, over the range of sizes, weight kinds and modes such programs use.

A case is a dict of plain values.  `listed()` names twelve; `draw(rng)` makes another one of the same
ranges; `prepare(case, seed)` makes what the program holds before the call (weights on the device in the
bundle layouts, registered; activations; a decoder; a recorded graph), `run(state)` is one pass through the
public entry points, `work(case)` the bytes and operations the pass cannot do without, and
`tolerance(case)` how far two correct implementations may lie apart.

Kinds of case:

  layer   the seven projections of one decoder layer, `rows` rows of activations each, in one
          linear_batch call: rows = 1 is a decode step's use, 2 to 15 a few sequences decoded together,
          16 and more a batch or a prompt (the matrix-core GEMM).
  sweep   every projection of a model and its lm_head for one token, replayed as a graph: what a host that
          keeps its own attention and norm kernels has the library do per token.
  head    the lm_head with the greedy token behind it.
  decode  `tokens` greedy steps of the device decoder from position `pos` on: a recorded graph per step, or
          (stream) plain launches with every token read back as it comes, as a chat loop that prints does.
  prompt  `tokens` prompt tokens at once at positions pos0 .. , up to the first answer token: time to first
          token of a new conversation (pos0 = 0) or of its next turn (pos0 > 0).

Weights are N(0, 0.02) rounded to fp16 and quantised as the bundle writers do, activations N(0, 1), norms
1 + N(0, 0.02), biases N(0, 0.02), tokens uniform; the lm_head is the embedding table, quantised (the
models tie the two).
"""
import importlib
import math

import torch

mil = importlib.import_module("adreno-llms_amd")

# hidden, inter, query heads, key/value heads, head width, layers, vocabulary
MODELS = {
    "qwen2.5-0.5b": dict(hidden=896, inter=4864, n_heads=14, n_kv_heads=2, head_dim=64, n_layers=24, vocab=151936,
                         rms_eps=1e-6, rope_theta=1000000.0),
    "smollm2-135m": dict(hidden=576, inter=1536, n_heads=9, n_kv_heads=3, head_dim=64, n_layers=30, vocab=49152,
                         rms_eps=1e-5, rope_theta=100000.0),
    "smollm2-360m": dict(hidden=960, inter=2560, n_heads=15, n_kv_heads=5, head_dim=64, n_layers=32, vocab=49152,
                         rms_eps=1e-5, rope_theta=100000.0),
}
CONTEXT = 4096                       # positions a decoder is made for
PROJECTIONS = ("wq", "wk", "wv", "wo", "wgate", "wup", "wdown")


def listed():
    return [
        # the smallest use: one layer's fp16 projections for one token of the smallest model, launch latency all of it
        dict(name="layer_f16_135m_1", kind="layer", model="smollm2-135m", weights="f16", rows=1),
        # a batch of 16 conversations decoded together: weights streamed once for all rows
        dict(name="layer_int8_05b_16", kind="layer", model="qwen2.5-0.5b", weights="int8", rows=16),
        # the same layer for a 2048-token prompt: the matrix-core GEMM at its largest configured size
        dict(name="layer_int8_05b_2048", kind="layer", model="qwen2.5-0.5b", weights="int8", rows=2048),
        # one decode step's matmuls, 169 of them (the benchmark's headline workload)
        dict(name="sweep_int8_05b", kind="sweep", model="qwen2.5-0.5b", weights="int8"),
        # the largest single GEMV, nibble-packed, with the greedy token behind it
        dict(name="head_q4_05b", kind="head", model="qwen2.5-0.5b", weights="q4"),
        # an answer's first tokens: short context, the whole step on the device, one graph per token
        dict(name="decode_int8_05b_short", kind="decode", model="qwen2.5-0.5b", weights="int8", pos=23, tokens=32,
             splits=0, stream=False),
        # a chat loop that prints every token as it comes, fp16 weights, no graph
        dict(name="decode_f16_135m_chat", kind="decode", model="smollm2-135m", weights="f16", pos=201, tokens=16,
             splits=0, stream=True),
        # an answer far into a conversation, the default attention (bit for bit the reference's order)
        dict(name="decode_int8_05b_1900", kind="decode", model="qwen2.5-0.5b", weights="int8", pos=1900, tokens=8,
             splits=0, stream=False),
        # the same further on, Q4 weights, with the mode for long contexts
        dict(name="decode_q4_05b_3701_splits", kind="decode", model="qwen2.5-0.5b", weights="q4", pos=3701, tokens=8,
             splits=16, stream=False),
        # time to first token of a one-line question
        dict(name="prompt_f16_360m_37", kind="prompt", model="smollm2-360m", weights="f16", tokens=37, pos0=0),
        # a next turn: a few hundred tokens behind what the conversation has in its cache
        dict(name="prompt_q4_05b_300_at_900", kind="prompt", model="qwen2.5-0.5b", weights="q4", tokens=300, pos0=900),
        # a long document at once
        dict(name="prompt_int8_05b_2048", kind="prompt", model="qwen2.5-0.5b", weights="int8", tokens=2048, pos0=0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "sweep", "head", "decode", "decode", "decode", "prompt", "prompt", "prompt"])
    case = dict(kind=kind, model=rng.choice(sorted(MODELS)), weights=rng.choice(["f16", "int8", "q4"]))
    if kind == "layer":
        case["rows"] = _log_int(rng, 1, 2048)
    elif kind == "sweep":
        case["layers"] = rng.randint(6, MODELS[case["model"]]["n_layers"] - 1)   # a model of the same widths, less deep
    elif kind == "head":
        case["vocab"] = _log_int(rng, 32000, 150000)                              # vocabularies are of any size, odd ones too
    elif kind == "decode":
        case["pos"] = _log_int(rng, 8, 2500)
        case["tokens"] = 6 if case["pos"] >= 1200 else 8 if case["pos"] >= 400 else rng.randint(8, 20)
        case["splits"] = rng.choice([0, 0, 8, 16, 32]) if case["pos"] >= 150 else 0
        case["stream"] = rng.random() < 0.3
    else:
        case["tokens"] = _log_int(rng, 8, 1500)
        case["pos0"] = rng.choice([0, 0, rng.randint(1, 1500)]) if case["tokens"] <= 600 else 0
    return case


# ---- what a program holds before the call ------------------------------------------------------------

_queue = None


def queue():
    """The program's one stream."""
    global _queue
    if _queue is None:
        assert mil.lib().mi_init(0) == 1
        _queue = mil.Queue()
    return _queue


class _Maker:
    """Seeded tensors on the GPU, handed over in the library's own device buffers."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, *shape, sigma=1.0, mean=0.0):
        return (torch.randn(shape, generator=self.gen, device="cuda") * sigma + mean).half()

    @staticmethod
    def buffer(t):
        t = t.contiguous()
        n = t.numel() * t.element_size()
        b = mil.Buffer(n)
        assert mil.lib().mi_memcpy_d2d(b.ptr, t.data_ptr(), n, None)
        return b

    def vector(self, n, mean=0.0):
        return self.buffer(self.normal(n, sigma=0.02, mean=mean))

    def weight(self, kind, w, keep):
        """fp16 matrix w in the bundle layout of `kind`, registered; keep receives the buffers."""
        n, k = w.shape
        if kind == "f16":
            keep.append(self.buffer(w))
            return keep[-1]
        f = w.float()
        if kind == "int8":
            scale = (f.abs().amax(1, keepdim=True) / 127).half()
            q = torch.round(f / scale.float()).clamp_(-127, 127).to(torch.int8)
        else:
            f = f.view(n, k // 32, 32)
            scale = (f.abs().amax(2, keepdim=True) / 7).half()
            q = (torch.round(f / scale.float()).clamp_(-8, 7) + 8).to(torch.uint8).view(n, k // 2, 2)
            q = q[:, :, 0] | (q[:, :, 1] << 4)
        wb, sb = self.buffer(q), self.buffer(scale)
        keep += [wb, sb]
        register = mil.nnopt_register_int8_weight if kind == "int8" else mil.nnopt_register_q4_weight
        assert register(wb, sb, n, k)
        return wb


def _shapes(cfg):
    qd, kvd = cfg["n_heads"] * cfg["head_dim"], cfg["n_kv_heads"] * cfg["head_dim"]
    h, i = cfg["hidden"], cfg["inter"]
    return dict(wq=(qd, h), wk=(kvd, h), wv=(kvd, h), wo=(h, qd), wgate=(i, h), wup=(i, h), wdown=(h, i))


def _layer_calls(make, cfg, weights, rows, keep, outs):
    """The seven calls of a layer: q, k, v from one input, o, gate and up from one input, down."""
    shapes, calls, inputs = _shapes(cfg), [], {}
    for name in PROJECTIONS:
        n, k = shapes[name]
        source = {"wk": "wq", "wv": "wq", "wup": "wgate"}.get(name, name)
        if source not in inputs:
            inputs[source] = make.buffer(make.normal(rows, k))
            keep.append(inputs[source])
        w = make.weight(weights, make.normal(n, k, sigma=0.02), keep)
        calls.append((rows, n, k, inputs[source], w, outs[name].data_ptr()))
    return calls


class _DeviceArray:
    """n fp16 values of memory that belongs to a decoder, in the form torch makes a tensor of."""

    def __init__(self, dec, ptr, n):
        self.dec = dec
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<f2", data=(ptr, False), version=2)


def _view(dec, ptr, n):
    """The decoder's own buffer as a tensor, which keeps the decoder alive for as long as it is held itself."""
    t = torch.as_tensor(_DeviceArray(dec, ptr, n), device="cuda")
    t.decoder = dec
    return t


def _decoder(make, cfg, weights, keep):
    layers, shapes = range(cfg["n_layers"]), _shapes(cfg)
    embed = make.normal(cfg["vocab"], cfg["hidden"], sigma=0.02)
    bufs = dict(embed=make.buffer(embed), final_norm=make.vector(cfg["hidden"], 1.0),
                lm_head=make.weight(weights, embed, keep),
                in_norm=[make.vector(cfg["hidden"], 1.0) for _ in layers],
                post_norm=[make.vector(cfg["hidden"], 1.0) for _ in layers],
                bq=[make.vector(shapes["wq"][0]) for _ in layers], bk=[make.vector(shapes["wk"][0]) for _ in layers],
                bv=[make.vector(shapes["wv"][0]) for _ in layers])
    for name in PROJECTIONS:
        bufs[name] = [make.weight(weights, make.normal(*shapes[name], sigma=0.02), keep) for _ in layers]
    torch.cuda.synchronize()
    return mil.Decoder(dict(cfg, max_pos=CONTEXT), bufs)


def _fill_cache(dec, tokens):
    """Keys and values of positions 0 .. len(tokens) - 1, as single-token steps leave them bit for bit (the
    projections as rows of GEMV), so that what is decoded behind them can be compared bit for bit."""
    q = queue()
    assert mil.lib().mi_stream_set_modes(q.handle, -1, 1)
    assert dec.prefill(q, tokens)
    q.finish()
    assert mil.lib().mi_stream_set_modes(q.handle, -1, -1)


def _tokens(make, cfg, n):
    return torch.randint(0, cfg["vocab"], (n,), generator=make.gen, device="cuda").tolist()


def _config(case):
    """The model of a case; a sweep may be of fewer layers, an lm_head of another vocabulary."""
    cfg = dict(MODELS[case["model"]])
    cfg["n_layers"], cfg["vocab"] = case.get("layers", cfg["n_layers"]), case.get("vocab", cfg["vocab"])
    return cfg


def prepare(case, seed):
    q, cfg, make, keep = queue(), _config(case), _Maker(seed), []
    kind, weights = case["kind"], case["weights"]
    state = dict(kind=kind, keep=keep)
    half = lambda *shape: torch.zeros(shape, dtype=torch.float16, device="cuda")  # noqa: E731
    shapes = _shapes(cfg)
    if kind == "layer":
        rows = case["rows"]
        outs = {name: half(rows, shapes[name][0]) for name in PROJECTIONS}
        state.update(outs=outs, calls=mil.make_calls(_layer_calls(make, cfg, weights, rows, keep, outs)))
    elif kind == "sweep":
        widths = [shapes[name][0] for name in PROJECTIONS]
        flat, logits = half(cfg["n_layers"], sum(widths)), half(cfg["vocab"])
        calls = []
        for layer in range(cfg["n_layers"]):
            outs = dict(zip(PROJECTIONS, torch.split(flat[layer], widths)))
            calls += _layer_calls(make, cfg, weights, 1, keep, outs)
        x = make.buffer(make.normal(1, cfg["hidden"]))
        keep.append(x)
        head = make.weight(weights, make.normal(cfg["vocab"], cfg["hidden"], sigma=0.02), keep)
        calls.append((1, cfg["vocab"], cfg["hidden"], x, head, logits.data_ptr()))
        arr = mil.make_calls(calls)
        torch.cuda.synchronize()
        assert mil.linear_batch(q, arr) == len(arr)      # first use of the kernels, outside the recording
        q.finish()
        with mil.Graph(q) as graph:
            assert mil.linear_batch(q, arr) == len(arr)
        state.update(graph=graph, outs=dict(projections=flat, logits=logits), calls=arr)
    elif kind == "head":
        logits, token = half(cfg["vocab"]), torch.zeros(1, dtype=torch.int32, device="cuda")
        x = make.buffer(make.normal(1, cfg["hidden"]))
        w = make.weight(weights, make.normal(cfg["vocab"], cfg["hidden"], sigma=0.02), keep)
        state.update(n=cfg["vocab"], k=cfg["hidden"], x=x, w=w, outs=dict(logits=logits, token=token))
    else:
        dec = _decoder(make, cfg, weights, keep)
        if kind == "decode":
            ids = _tokens(make, cfg, case["pos"] + 1)
            _fill_cache(dec, ids[:-1])
            if case["splits"]:
                assert dec.set_attention_splits(case["splits"])
            assert dec.reset(q, case["pos"], ids[-1]) and dec.step(q)
            q.finish()
            graph = None
            if not case["stream"]:
                with mil.Graph(q) as graph:
                    assert dec.step(q)
            state.update(pos=case["pos"], first=ids[-1], steps=case["tokens"], graph=graph)
        else:
            ids = _tokens(make, cfg, case["pos0"] + case["tokens"])
            if case["pos0"]:
                _fill_cache(dec, ids[:case["pos0"]])
            assert dec.reserve_prompt(q, case["tokens"])
            state.update(ids=ids[case["pos0"]:], pos0=case["pos0"])
        hidden = mil.lib().mi_decoder_buffer(dec.handle, 0)
        state.update(dec=dec, outs=dict(logits=_view(dec, dec.logits_ptr, cfg["vocab"]),
                                        hidden=_view(dec, hidden, cfg["hidden"])))
    torch.cuda.synchronize()
    return state


# ---- one pass --------------------------------------------------------------------------------------

def run(state):
    q, kind, outs = queue(), state["kind"], state["outs"]
    if kind == "layer":
        assert mil.linear_batch(q, state["calls"]) == len(state["calls"])
        return outs
    if kind == "sweep":
        state["graph"].launch()
        return outs
    if kind == "head":
        assert mil.pytorch_linear_argmax(q, state["n"], state["k"], state["x"], state["w"], outs["logits"].data_ptr(),
                                         outs["token"].data_ptr())
        return outs
    dec = state["dec"]
    if kind == "prompt":
        assert dec.prefill(q, state["ids"], state["pos0"])
        return dict(outs, position_and_token=list(dec.read(q)))
    assert dec.reset(q, state["pos"], state["first"])
    if state["graph"] is None:
        tokens = []
        for _ in range(state["steps"]):
            assert dec.step(q)
            tokens.append(dec.read(q)[1])
        return dict(outs, tokens=tokens)
    for _ in range(state["steps"]):
        state["graph"].launch()
    return dict(outs, position_and_token=list(dec.read(q)))


# ---- what a pass cannot do without -----------------------------------------------------------------

def _weight_bytes(weights, n, k):
    return {"f16": 2 * n * k, "int8": n * k + 2 * n, "q4": n * k // 2 + 2 * n * (k // 32)}[weights]


def work(case):
    cfg, weights = _config(case), case["weights"]
    shapes, head = list(_shapes(cfg).values()), (cfg["vocab"], cfg["hidden"])
    layer_bytes = sum(_weight_bytes(weights, n, k) for n, k in shapes)
    layer_macs = sum(n * k for n, k in shapes)
    head_bytes = _weight_bytes(weights, *head) + 2 * sum(head)
    qd, kvd, layers = shapes[0][0], shapes[1][0], cfg["n_layers"]
    kind = case["kind"]
    # inputs of a layer's projections (q | k | v and gate | up share theirs) and their outputs, per row
    row_bytes = 2 * (2 * cfg["hidden"] + qd + cfg["inter"]) + 2 * sum(n for n, _ in shapes)
    if kind == "layer":
        rows = case["rows"]
        return dict(bytes=layer_bytes + rows * row_bytes, flops=2 * rows * layer_macs)
    if kind == "sweep":
        return dict(bytes=layers * (layer_bytes + row_bytes) + head_bytes, flops=2 * (layers * layer_macs + head[0] * head[1]))
    if kind == "head":
        return dict(bytes=head_bytes + 4, flops=2 * head[0] * head[1])
    if kind == "decode":
        first, n = case["pos"], case["tokens"]
        keys = sum(range(first + 1, first + n + 1))               # keys (and values) seen by the n tokens together
        return dict(bytes=n * (layers * layer_bytes + head_bytes) + layers * 2 * 2 * kvd * keys,
                    flops=2 * n * (layers * layer_macs + head[0] * head[1]) + 4 * layers * qd * keys)
    first, n = case["pos0"], case["tokens"]
    keys = sum(range(first + 1, first + n + 1))
    return dict(bytes=layers * (layer_bytes + 2 * 2 * kvd * (first + n)) + head_bytes + 2 * n * cfg["hidden"],
                flops=2 * (n * layers * layer_macs + head[0] * head[1]) + 4 * layers * qd * keys)


def tolerance(case):
    kind, weights = case["kind"], case["weights"]
    # One row, fp16 and int8 weights: the library promises the reference's order of operations, bit for bit.
    if weights != "q4" and (kind in ("sweep", "head") or (kind == "layer" and case["rows"] == 1) or
                            (kind == "decode" and not case["splits"])):
        return "exact"
    # Projections whose fp32 sums may run in any order, rounded to fp16 once: a few outputs in a thousand land
    # on the neighbouring fp16 number.  Measured between the matrix-core GEMM (Q4: also the throughput GEMV) and
    # the reference's order: rel 1.1e-5 (Q4: 4.9e-5), largest difference 1e-3 of the value (one fp16 step).
    if kind in ("layer", "sweep", "head"):
        return {"rel": 2e-4 if weights == "q4" else 5e-5, "max": 4e-3}
    # The same through all layers of a model: rel 2.5e-3 to 2.9e-3, largest 1.4e-2, for prompts of 300 to 2048 tokens
    # and for steps with the keys split, against the reference's order throughout.
    return {"rel": 1e-2, "max": 6e-2}
