"""The workloads this framework's speed is measured on: what a serving engine asks of it for one
batch, through the public entry points it calls (`Int8Linear`, `Int8GluMLP`, `Int8RMSNormQuant`,
`PackedBf16Linear`, `ops.paged_attention_forward`, `DecodeRunner`).

Sizes are those of the Llama-3-8B linears (hidden 4096, intermediate 14336, 32 query over 8 K/V
heads of 128, vocabulary 128256) and of Llama-3.2-3B, the default model of `ModelConfig` (hidden
3072, intermediate 8192, 24 query heads over 8). An engine iteration holds at most 64 sequences
and 4096 prompt tokens, prompts are cut into chunks of at most 2048 tokens, and the K/V pool has
16-slot blocks.

A case is a dict with a `kind`:
  * "linear": one `Int8Linear` call, m rows of k inputs to n outputs, in a mode: "int8"
    (weight-only, bf16 activations) or "w8a8" (activations quantized per token);
  * "mlp": one `Int8GluMLP` call (gate, up, SiLU-mul, down); with `norm` the `Int8RMSNormQuant`
    before it, as the W8A8 decoder layer runs them;
  * "head": the bf16 lm_head on m rows;
  * "attention": one paged attention call of `decodes` sequences with one query row each and
    `chunks` prompt chunks of up to `chunk` tokens, behind up to `ctx` cached positions;
  * "step": a whole decode step of `batch` sequences (embedding to logits) behind `ctx` cached
    positions, replayed from the graph it was captured into, as the engine runs decode.
"""

from __future__ import annotations

import math
import random

import torch

import __graft_entry__

D = 128  # head size
BLOCK = 16  # slots of a K/V block
VOCAB = 128256

# (k, n) of the projections: q/k/v stacked, o, down; the last two are generic.
PROJECTIONS = [(4096, 6144), (4096, 4096), (14336, 4096), (3072, 5120), (3072, 3072), (8192, 3072),
               (2048, 2048), (4096, 1024)]
MLPS = [(4096, 14336), (3072, 8192), (2048, 8192)]
HEADS = [(32, 8), (24, 8)]


def listed():
    return [
        # One sequence decoding, called from the host: the smallest call.
        dict(name="decode qkv 1", kind="linear", mode="int8", m=1, k=4096, n=6144),
        # A middling decode batch over the narrowest projection.
        dict(name="decode o 32", kind="linear", mode="int8", m=32, k=4096, n=4096),
        # The W8A8 mode's deepest projection at a small decode batch: bf16 rows arrive and are
        # quantized on the way.
        dict(name="decode down w8a8 16", kind="linear", mode="w8a8", m=16, k=14336, n=4096),
        # The MLP of a full decode batch.
        dict(name="decode mlp 64", kind="mlp", mode="int8", norm=False, m=64, k=4096, i=14336),
        # Next-token logits of a full decode batch.
        dict(name="head 64", kind="head", m=64, k=4096, n=VOCAB),
        # A prompt chunk of the longest length the engine cuts, weight-only.
        dict(name="prefill qkv 2048", kind="linear", mode="int8", m=2048, k=4096, n=6144),
        # A short prompt of odd length through the 3B model's MLP.
        dict(name="prefill mlp 417", kind="mlp", mode="int8", norm=False, m=417, k=3072, i=8192),
        # A full iteration's prompt tokens through the W8A8 MLP block with its norm: the largest.
        dict(name="prefill mlp w8a8 4096", kind="mlp", mode="w8a8", norm=True, m=4096, k=4096,
             i=14336),
        # Attention of a full decode batch over contexts of different lengths.
        dict(name="attention decode 64", kind="attention", h=32, h_kv=8, decodes=64, chunks=0,
             chunk=0, ctx=2048, lens=1),
        # Attention of fresh prompts.
        dict(name="attention prefill", kind="attention", h=32, h_kv=8, decodes=0, chunks=3,
             chunk=2048, ctx=0, lens=2),
        # Continuous batching: a later chunk of one prompt beside decoding sequences, 24 heads
        # over 8.
        dict(name="attention mixed", kind="attention", h=24, h_kv=8, decodes=40, chunks=1,
             chunk=1024, ctx=2048, lens=3),
        # A whole decode step of a full batch at a context of 1024, four layers.
        dict(name="step 64", kind="step", batch=64, ctx=1024, layers=4),
    ]


def _log(rng: random.Random, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["linear"] * 4 + ["mlp"] * 3 + ["head"] + ["attention"] * 4 + ["step"])
    if kind == "linear":
        m = _log(rng, 1, 4096)
        k, n = rng.choice(PROJECTIONS)
        if rng.random() < 0.3:  # a projection of no particular model, any row count
            k, n = 16 * _log(rng, 32, 768), _log(rng, 500, 12000)
        return dict(kind=kind, mode=rng.choice(["int8", "w8a8"]), m=m, k=k, n=n)
    if kind == "mlp":
        mode = rng.choice(["int8", "w8a8"])
        k, i = rng.choice(MLPS)
        return dict(kind=kind, mode=mode, norm=mode == "w8a8",
                    m=_log(rng, 1, 4096 if mode == "w8a8" else 2048), k=k, i=i)
    if kind == "head":
        return dict(kind=kind, m=_log(rng, 1, 64), k=rng.choice([4096, 3072]), n=VOCAB)
    if kind == "attention":
        h, h_kv = rng.choice(HEADS)
        what = rng.choice(["decode", "prefill", "mixed"])
        lens = rng.randrange(1 << 20)
        if what == "decode":
            return dict(kind=kind, h=h, h_kv=h_kv, decodes=_log(rng, 1, 64), chunks=0, chunk=0,
                        ctx=_log(rng, 64, 4096), lens=lens)
        if what == "prefill":
            chunk = _log(rng, 32, 2048)
            return dict(kind=kind, h=h, h_kv=h_kv, decodes=0,
                        chunks=rng.randint(1, max(1, min(8, 4096 // chunk))), chunk=chunk,
                        ctx=rng.choice([0, 0, _log(rng, 64, 2048)]), lens=lens)
        return dict(kind=kind, h=h, h_kv=h_kv, decodes=_log(rng, 1, 63), chunks=1,
                    chunk=_log(rng, 16, 1024), ctx=_log(rng, 64, 2048), lens=lens)
    return dict(kind=kind, batch=_log(rng, 1, 64), ctx=_log(rng, 100, 1024),
                layers=rng.randint(2, 4))


# ---- inputs ------------------------------------------------------------------------------------


def _gen(seed: int, what: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(16 * seed + what)


def _randn(g: torch.Generator, *shape: int) -> torch.Tensor:
    return torch.randn(*shape, generator=g, device="cuda")


def _rows(case, seed: int, k: int) -> torch.Tensor:
    """bf16 activations ~ N(0, 1); in the W8A8 mode 0.1 % of the columns are 20 times larger, the
    outlier channels that mode meets."""
    x = _randn(_gen(seed, 0), case["m"], k)
    if case.get("mode") == "w8a8":
        cols = torch.randperm(k, generator=_gen(seed, 1), device="cuda")[:max(1, round(0.001 * k))]
        x[:, cols] *= 20.0
    return x.to(torch.bfloat16)


def _quantized(w: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """Per-output-channel symmetric int8 of an fp32 (N, K) weight, and its scales."""
    s = w.abs().amax(1) / 127.0
    q = torch.clamp(torch.round(w / s[:, None]), -127, 127).to(torch.int8)
    return q, s


def _weight(seed: int, what: int, n: int, k: int) -> tuple[torch.Tensor, torch.Tensor]:
    return _quantized(0.02 * _randn(_gen(seed, what), n, k))


def _mlp_weights(case, seed: int):
    q, s = _weight(seed, 2, 2 * case["i"], case["k"])  # [gate; up]
    qd, sd = _weight(seed, 3, case["k"], case["i"])
    return q, s, qd, sd


def _norm_weight(case, seed: int) -> torch.Tensor:
    return (1.0 + 0.1 * _randn(_gen(seed, 4), case["k"])).to(torch.bfloat16)


class _Norm:
    """What `Int8RMSNormQuant` takes over from a decoder layer's norm."""

    def __init__(self, weight: torch.Tensor) -> None:
        self.weight = torch.nn.Parameter(weight, requires_grad=False)
        self.variance_epsilon = 1e-5


def _entries(case) -> list[tuple[int, int]]:
    """(query rows, context length) of each entry of an attention call."""
    r = random.Random(case["lens"])
    got = []
    for _ in range(case["chunks"]):
        rows = r.randint(max(1, (3 * case["chunk"]) // 5), case["chunk"])
        got.append((rows, rows + (r.randint(case["ctx"] // 2, case["ctx"]) if case["ctx"] else 0)))
    for _ in range(case["decodes"]):
        got.append((1, r.randint(max(1, case["ctx"] // 8), case["ctx"])))
    return got


def _attention_inputs(case, seed: int):
    """q, k_pool, v_pool, block_table, context_len, query_offset, q_start, q_len: every entry owns
    shuffled blocks of one pool, whose last block is nobody's."""
    entries = _entries(case)
    need = [-(-ctx // BLOCK) for _, ctx in entries]
    perm = torch.randperm(sum(need), generator=torch.Generator().manual_seed(seed))
    table = torch.zeros(len(entries), max(need), dtype=torch.int32)
    at = 0
    for e, n in enumerate(need):
        table[e, :n] = perm[at:at + n]
        at += n
    rows = [q for q, _ in entries]
    start = [sum(rows[:e]) for e in range(len(rows))]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    q = _randn(_gen(seed, 0), case["h"], sum(rows), D).to(torch.bfloat16)
    pool = (sum(need) + 1, BLOCK, case["h_kv"], D)
    k = _randn(_gen(seed, 1), *pool).to(torch.bfloat16)
    v = _randn(_gen(seed, 2), *pool).to(torch.bfloat16)
    return (q, k, v, table.cuda(), i32([c for _, c in entries]), i32([c - n for n, c in entries]),
            i32(start), i32(rows))


HIDDEN, INTER, H, H_KV, EPS, THETA = 4096, 14336, 32, 8, 1e-5, 500000.0


def _model_weights(case, seed: int):
    """(name, bf16 tensor) of every parameter of the decoder, in order."""
    g = _gen(seed, 5)
    mat = lambda n, k: (0.02 * _randn(g, n, k)).to(torch.bfloat16)  # noqa: E731
    norm = lambda: (1.0 + 0.1 * _randn(g, HIDDEN)).to(torch.bfloat16)  # noqa: E731
    yield "model.embed_tokens.weight", mat(VOCAB, HIDDEN)
    for i in range(case["layers"]):
        p = f"model.layers.{i}."
        yield p + "self_attn.q_proj.weight", mat(H * D, HIDDEN)
        yield p + "self_attn.k_proj.weight", mat(H_KV * D, HIDDEN)
        yield p + "self_attn.v_proj.weight", mat(H_KV * D, HIDDEN)
        yield p + "self_attn.o_proj.weight", mat(HIDDEN, H * D)
        yield p + "mlp.gate_proj.weight", mat(INTER, HIDDEN)
        yield p + "mlp.up_proj.weight", mat(INTER, HIDDEN)
        yield p + "mlp.down_proj.weight", mat(HIDDEN, INTER)
        yield p + "input_layernorm.weight", norm()
        yield p + "post_attention_layernorm.weight", norm()
    yield "model.norm.weight", norm()
    yield "lm_head.weight", mat(VOCAB, HIDDEN)


def _step_cache(case, seed: int, layer: int):
    """bf16 K and V (batch, heads, ctx, D) of a layer's cached positions."""
    g = _gen(seed, 6)
    g.manual_seed(g.initial_seed() + 1000 * layer)
    shape = (case["batch"], H_KV, case["ctx"], D)
    return _randn(g, *shape).to(torch.bfloat16), _randn(g, *shape).to(torch.bfloat16)


def _step_tokens(case, seed: int) -> torch.Tensor:
    return torch.randint(0, VOCAB, (case["batch"],), generator=_gen(seed, 7), device="cuda")


def _prepare_step(case, seed: int):
    pkg = __graft_entry__.load_package()
    from llm_serving_engine_amd.decode_step import DecodeRunner, random_llama

    model = random_llama(case["layers"], 0, torch.device("cuda"))
    params = dict(model.named_parameters())
    with torch.no_grad():
        for name, w in _model_weights(case, seed):
            params[name].copy_(w)
    runner = DecodeRunner(model, case["batch"], case["ctx"] + BLOCK)
    runner.quantize("int8")
    for i in range(case["layers"]):
        k, v = _step_cache(case, seed, i)
        runner.k_cache[i][:, :, :case["ctx"]] = k
        runner.v_cache[i][:, :, :case["ctx"]] = v
    runner.enable_paged(BLOCK, seed)
    runner.use("int8")
    runner.use_attention("paged")
    tokens = _step_tokens(case, seed)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        runner.step(tokens, case["ctx"])
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        logits = runner.step(tokens, case["ctx"])
    return dict(pkg=pkg, graph=graph, runner=runner, tokens=tokens, logits=logits)


def prepare(case, seed):
    if case["kind"] == "step":
        return _prepare_step(case, seed)
    pkg = __graft_entry__.load_package()
    from llm_serving_engine_amd import int8_linear as il

    if case["kind"] == "linear":
        q, s = _weight(seed, 2, case["n"], case["k"])
        return dict(mod=il.Int8Linear.from_quantized(q, s, case["mode"]),
                    x=_rows(case, seed, case["k"]))
    if case["kind"] == "mlp":
        q, s, qd, sd = _mlp_weights(case, seed)
        mlp = il.Int8GluMLP(il.Int8GateUp.from_quantized(q, s, case["mode"]),
                            il.Int8Linear.from_quantized(qd, sd, case["mode"]))
        mod = mlp
        if case["norm"]:
            mod = torch.nn.Sequential(il.Int8RMSNormQuant(_Norm(_norm_weight(case, seed))), mlp)
        return dict(mod=mod, x=_rows(case, seed, case["k"]))
    if case["kind"] == "head":
        lin = torch.nn.Linear(case["k"], case["n"], bias=False, device="cuda",
                              dtype=torch.bfloat16)
        with torch.no_grad():
            lin.weight.copy_(0.02 * _randn(_gen(seed, 2), case["n"], case["k"]))
        return dict(mod=il.PackedBf16Linear.from_linear(lin), x=_rows(case, seed, case["k"]))
    return dict(attend=pkg.ops.paged_attention_forward, args=_attention_inputs(case, seed),
                most=max(q for q, _ in _entries(case)))


def run(state):
    if "graph" in state:
        state["graph"].replay()
        runner = state["runner"]
        # The step's logits, and the pools that it wrote its K and V rows to.
        return [state["logits"], *runner.k_pool, *runner.v_pool]
    if "attend" in state:
        return state["attend"](*state["args"], BLOCK, state["most"])
    with torch.no_grad():
        return state["mod"](state["x"])


# ---- what a pass cannot do without -------------------------------------------------------------


def _linear_work(case, m: int, k: int, n: int) -> tuple[float, float]:
    return k * n + 4 * n + 2 * m * k + 2 * m * n, 2 * m * n * k


def work(case):
    if case["kind"] == "linear":
        b, f = _linear_work(case, case["m"], case["k"], case["n"])
        return dict(bytes=b, flops=f)
    if case["kind"] == "mlp":
        m, k, i = case["m"], case["k"], case["i"]
        return dict(bytes=3 * k * i + 4 * (2 * i + k) + 4 * m * k, flops=6 * m * k * i)
    if case["kind"] == "head":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(bytes=2 * (k * n + m * k + m * n), flops=2 * m * n * k)
    if case["kind"] == "attention":
        entries = _entries(case)
        rows = sum(q for q, _ in entries)
        kv = sum(c for _, c in entries) * case["h_kv"] * D * 4
        # Query row r of an entry sees the positions up to its own.
        seen = sum(q * (c - q) + q * (q + 1) // 2 for q, c in entries)
        return dict(bytes=kv + 4 * case["h"] * rows * D, flops=4 * D * case["h"] * seen)
    m, c = case["batch"], case["ctx"] + 1
    params = case["layers"] * ((H + 2 * H_KV) * D * HIDDEN + H * D * HIDDEN + 3 * HIDDEN * INTER)
    kv = case["layers"] * m * c * H_KV * D
    return dict(bytes=params + 2 * VOCAB * HIDDEN + 4 * kv + 2 * m * (VOCAB + HIDDEN),
                flops=2 * m * (params + VOCAB * HIDDEN) + 4 * kv * (H // H_KV))


def tolerance(case):
    if case["kind"] == "step":
        return dict(rel=0.03, max=0.2)
    if case["kind"] == "mlp":
        return dict(rel=0.01, max=0.1)
    if case["kind"] == "attention":
        return dict(rel=0.009, max=0.1)
    return dict(rel=0.007, max=0.02)


# ---- the same in 64 bits -----------------------------------------------------------------------


def _bf16(x: torch.Tensor) -> torch.Tensor:
    return x.to(torch.float32).to(torch.bfloat16).to(torch.float64)


def _product(mode: str, x: torch.Tensor, q: torch.Tensor, s: torch.Tensor) -> torch.Tensor:
    """x (fp64 holding bf16 values) times the quantized weight; in the W8A8 mode x is first put on
    its row's int8 grid, which is what that mode means."""
    if mode == "w8a8":
        x32 = x.float()
        sx = x32.abs().amax(1, keepdim=True) / 127.0
        sx = torch.where(sx > 0, sx, torch.ones_like(sx))
        x = torch.clamp(torch.round(x32 / sx), -127, 127).double() * sx.double()
    return (x @ q.double().t().contiguous()) * s.double()


def _silu(x: torch.Tensor) -> torch.Tensor:
    return x / (1.0 + torch.exp(-x))


def _rms(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, first: int) -> torch.Tensor:
    """q (rows, D) at positions `first` on, k and v (positions, D)."""
    score = (q @ k.t().contiguous()) / math.sqrt(D)
    at = torch.arange(first, first + q.shape[0], device=q.device)[:, None]
    hide = torch.arange(k.shape[0], device=q.device)[None, :] > at
    return torch.softmax(score.masked_fill(hide, -math.inf), -1) @ v


def _exact_attention(case, seed: int) -> torch.Tensor:
    q, k, v, table, *_ = _attention_inputs(case, seed)
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    group, at = case["h"] // case["h_kv"], 0
    for e, (rows, ctx) in enumerate(_entries(case)):
        blocks = table[e, :-(-ctx // BLOCK)].long()
        ke = k[blocks].reshape(-1, case["h_kv"], D)[:ctx].double()
        ve = v[blocks].reshape(-1, case["h_kv"], D)[:ctx].double()
        for h in range(case["h"]):
            out[h, at:at + rows] = _attend(q[h, at:at + rows].double(), ke[:, h // group].contiguous(),
                                           ve[:, h // group].contiguous(), ctx - rows)
        at += rows
    return out


def _rope(x: torch.Tensor, at: int) -> torch.Tensor:
    """x (..., D) rotated to position `at`."""
    half = torch.arange(0, D, 2, device=x.device, dtype=torch.float64) / D
    angle = at / THETA ** half
    cos, sin = torch.cos(angle).repeat(2), torch.sin(angle).repeat(2)
    return x * cos + torch.cat([-x[..., D // 2:], x[..., :D // 2]], -1) * sin


def _exact_step(case, seed: int) -> list:
    w = dict(_model_weights(case, seed))
    m, at = case["batch"], case["ctx"]

    def lin(x, *names):
        q, s = _quantized(torch.cat([w[n] for n in names]).float())
        return _product("int8", x, q, s)

    x = w["model.embed_tokens.weight"][_step_tokens(case, seed)].double()
    for i in range(case["layers"]):
        p = f"model.layers.{i}."
        h = _rms(x, w[p + "input_layernorm.weight"])
        qkv = lin(h, *(p + f"self_attn.{n}_proj.weight" for n in "qkv")).reshape(m, -1, D)
        q, k = _rope(qkv[:, :H], at), _rope(qkv[:, H:H + H_KV], at)
        v = qkv[:, H + H_KV:]
        ck, cv = _step_cache(case, seed, i)
        keys = torch.cat([ck.double(), k[:, :, None]], 2)
        vals = torch.cat([cv.double(), v[:, :, None]], 2)
        out = torch.empty(m, H, D, dtype=torch.float64, device="cuda")
        for b in range(m):
            for g in range(H_KV):
                rows = slice(g * (H // H_KV), (g + 1) * (H // H_KV))
                score = (q[b, rows] @ keys[b, g].t().contiguous()) / math.sqrt(D)
                out[b, rows] = torch.softmax(score, -1) @ vals[b, g]
        x = x + lin(out.reshape(m, H * D), p + "self_attn.o_proj.weight")
        h = _rms(x, w[p + "post_attention_layernorm.weight"])
        gu = lin(h, p + "mlp.gate_proj.weight", p + "mlp.up_proj.weight")
        x = x + lin(_silu(gu[:, :INTER]) * gu[:, INTER:], p + "mlp.down_proj.weight")
    x = _rms(x, w["model.norm.weight"])
    logits = x @ w["lm_head.weight"].double().t().contiguous()
    return [logits] + [None] * (2 * case["layers"])


@torch.no_grad()
def exact(case, seed):
    if case["kind"] == "step":
        return _exact_step(case, seed)
    if case["kind"] == "attention":
        return _exact_attention(case, seed)
    if case["kind"] == "head":
        w = (0.02 * _randn(_gen(seed, 2), case["n"], case["k"])).to(torch.bfloat16)
        return _rows(case, seed, case["k"]).double() @ w.double().t().contiguous()
    x = _rows(case, seed, case["k"]).double()
    if case["kind"] == "linear":
        return _product(case["mode"], x, *_weight(seed, 2, case["n"], case["k"]))
    q, s, qd, sd = _mlp_weights(case, seed)
    if case["norm"]:
        r = torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS)
        x = _bf16(_bf16(x * r) * _norm_weight(case, seed).double())
    gu = _product(case["mode"], x, q, s)
    h = _silu(gu[:, :case["i"]]) * gu[:, case["i"]:]
    if case["mode"] == "w8a8":
        h = _bf16(h)
    return _product(case["mode"], h, qd, sd)
