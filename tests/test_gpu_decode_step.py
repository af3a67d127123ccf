"""Config 4 at small scale on the GPU: the decode-step runner (the reference's fused decoder path
with the int8 linears swapped in) against the same runner on the reference's bf16 linears."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def runner(pkg, dev):
    from llm_serving_engine_amd.decode_step import DecodeRunner, random_llama

    model = random_llama(2, seed=11, device=dev)
    r = DecodeRunner(model, batch=16, capacity=40)
    gen = torch.Generator().manual_seed(12)
    r.prefill(torch.randint(0, model.config.vocab_size, (16, 32), generator=gen).to(dev), chunk=4)
    return r


def test_int8_step_tracks_the_bf16_reference(runner, dev):
    gen = torch.Generator().manual_seed(13)
    vocab = runner.model.config.vocab_size
    tok = torch.randint(0, vocab, (16,), generator=gen).to(dev)
    runner.use("bf16")
    ref, inputs = [], []
    for t in range(3):
        inputs.append(tok)
        logits = runner.step(tok, 32 + t).float()
        ref.append(logits)
        tok = logits.argmax(-1)
    runner.quantize("int8")
    runner.use("int8")
    matches = 0
    for t in range(3):
        logits = runner.step(inputs[t], 32 + t).float()
        rel = (logits - ref[t]).norm() / ref[t].norm()
        assert rel < 0.05, f"step {t}: logits differ by {rel:.3f} (relative norm)"
        matches += int((logits.argmax(-1) == ref[t].argmax(-1)).sum())
    assert matches >= 0.9 * 48, f"greedy match {matches}/48"


def test_int8_kernels_match_the_torch_restatement(runner, dev):
    """The same quantized weights through the HIP kernels and through an eager fp32 torch
    restatement: logits agree to bf16 rounding and fp32 order, and so do the greedy tokens."""
    if runner.int8 is None:
        runner.quantize("int8")
    gen = torch.Generator().manual_seed(14)
    tok = torch.randint(0, runner.model.config.vocab_size, (16,), generator=gen).to(dev)
    runner.use("int8-torch")
    ref = runner.step(tok, 35).float()
    runner.use("int8")
    got = runner.step(tok, 35).float()
    rel = (got - ref).norm() / ref.norm()
    assert rel < 1e-2, f"relative logit difference {rel:.4f}"
    assert int((got.argmax(-1) == ref.argmax(-1)).sum()) >= 15


def test_int8_linear_stack_replays_from_a_graph(runner, dev):
    """All projections of one step captured into one graph: every replay equals eager."""
    if runner.int8 is None:
        runner.quantize("int8")
    runner.use("int8")
    calls = runner.linear_calls(16)
    eager = [mod(x) for mod, x in calls]
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        outs = [mod(x) for mod, x in calls]
    for _ in range(3):
        g.replay()
        torch.cuda.synchronize()
        for a, b in zip(eager, outs):
            assert torch.equal(a, b)


def test_paged_attention_matches_the_torch_attention(runner, dev):
    """One int8 decode step through the HIP paged attention (shuffled 16-slot blocks) and through
    the fp32 torch attention over the contiguous cache: logits agree to the bf16 rounding of the
    probabilities, and so do the greedy tokens."""
    if runner.int8 is None:
        runner.quantize("int8")
    runner.use("int8")
    if runner.k_pool is None:
        runner.enable_paged()
    gen = torch.Generator().manual_seed(15)
    tok = torch.randint(0, runner.model.config.vocab_size, (16,), generator=gen).to(dev)
    runner.use_attention("torch")
    ref = runner.step(tok, 36).float()
    runner.use_attention("paged")
    got = runner.step(tok, 36).float()
    runner.use_attention("torch")
    rel = (got - ref).norm() / ref.norm()
    assert rel < 1e-2, f"relative logit difference {rel:.4f}"
    assert int((got.argmax(-1) == ref.argmax(-1)).sum()) >= 15


def test_whole_step_replays_from_a_graph(runner, dev):
    """The reference's graphed-decode invariant (tests/test_decode_graph.py:53-59: graphed ==
    eager) on the swapped path: one whole decode step (embedding to logits) with the int8 linears
    and the HIP paged attention, captured into a graph, equals the eager step bitwise on every
    replay, with eager steps in between. Each step writes the same K/V values at the same
    position, so every run sees the same state."""
    if runner.int8 is None:
        runner.quantize("int8")
    runner.use("int8")
    if runner.k_pool is None:
        runner.enable_paged()
    runner.use_attention("paged")
    gen = torch.Generator().manual_seed(16)
    tok = torch.randint(0, runner.model.config.vocab_size, (16,), generator=gen).to(dev)
    pos = 37
    eager = runner.step(tok, pos).clone()
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        runner.step(tok, pos)
    torch.cuda.current_stream().wait_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = runner.step(tok, pos)
    try:
        for i in range(3):
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, eager), f"replay {i}"
            again = runner.step(tok, pos)
            torch.cuda.synchronize()
            assert torch.equal(again, eager), f"eager after replay {i}"
    finally:
        runner.use_attention("torch")


@pytest.mark.parametrize("rows", [[4, 5, 6], torch.tensor([4, 5, 6])])
def test_indexed_rows_write_their_cache(runner, dev, rows):
    """Sequences given by index, whose cache rows are a copy and not a view: the same K/V writes and
    the same hidden states as the slice of them."""
    if runner.int8 is None:
        runner.quantize("int8")
    runner.use("int8")
    runner.use_attention("torch")
    gen = torch.Generator().manual_seed(17)
    tok = torch.randint(0, runner.model.config.vocab_size, (3, 1), generator=gen).to(dev)
    want = runner.forward(tok, 36, slice(4, 7))
    caches = [(c, c[4:7, :, 36].clone()) for c in (*runner.k_cache, *runner.v_cache)]
    for c, _ in caches:
        c[4:7, :, 36] = 0
    got = runner.forward(tok, 36, rows)
    assert torch.equal(got, want)
    for c, kv in caches:
        assert torch.equal(c[4:7, :, 36], kv)


@torch.no_grad()
def _unfused(r, tokens, start, rows):
    """`DecodeRunner.forward` spelled out with the reference's eager operations: each block's residual
    added before the next norm (decoder_hidden, model_runner.py:213-224)."""
    nseq, ntok = tokens.shape
    model = r.model.model
    r._rows, r._fused = rows, False
    if r.attention == "paged":
        r._plan = r._paged_plan(start, start + ntok, nseq, ntok)
    pos = torch.arange(start, start + ntok, device=tokens.device).repeat(nseq, 1)
    hidden = model.embed_tokens(tokens.reshape(1, -1))
    cos, sin = model.rotary_emb(hidden, pos.reshape(1, -1))
    for i, layer in enumerate(r.layers):
        normed = layer.input_layernorm(hidden)
        hidden = hidden + r._attend(i, normed, (cos[0], sin[0]), start, nseq, ntok)
        hidden = hidden + r._mlp(i, layer.post_attention_layernorm(hidden))
    return model.norm(hidden)


@pytest.mark.parametrize("attention", ["torch", "paged"])
@pytest.mark.parametrize("ntok", [1, 3])
def test_fused_kernels_against_the_eager_operations(runner, dev, attention, ntok):
    """A forward with the fused kernels and one of eager operations, written in the reference's order,
    from the same cache: the norms' sums of squares alone differ (in fp32), which moves few bf16
    roundings; a norm, residual, position or row taken from the wrong place changes everything."""
    runner.enable_paged()
    runner.use_attention(attention)
    try:
        runner.use("bf16")
        gen = torch.Generator().manual_seed(19)
        tok = torch.randint(0, runner.model.config.vocab_size, (5, ntok), generator=gen).to(dev)
        rows, at = slice(3, 8), slice(33, 33 + ntok)
        got = runner.forward(tok, 33, rows)
        assert runner._fused
        written = [c[rows, :, at].clone() for c in (*runner.k_cache, *runner.v_cache)]
        pools = [p.clone() for p in (*runner.k_pool, *runner.v_pool)]
        want = _unfused(runner, tok, 33, rows)
        rel = lambda a, b: float((a.float() - b.float()).norm() / b.float().norm())  # noqa: E731
        assert rel(got, want) < 0.01
        caches = [c[rows, :, at] for c in (*runner.k_cache, *runner.v_cache)]
        for layer, (a, b) in enumerate(zip(written, caches)):
            assert rel(a, b) < 0.01, f"cache {layer}"
        for layer, (a, b) in enumerate(zip(pools, (*runner.k_pool, *runner.v_pool))):
            assert rel(a, b) < 0.01, f"pool {layer}"
        assert rel(runner.lm_head()(got[0]), runner.lm_head()(want[0])) < 0.01
    finally:
        runner.use_attention("torch")


def test_a_norm_with_other_behaviour_is_called(runner, dev):
    """A norm whose forward was replaced runs, and so does a hook on every module."""
    runner.use("bf16")
    tok = torch.full((2, 1), 7, device=dev)
    norm, calls = runner.model.model.norm, []
    norm.forward = lambda x: torch.zeros_like(x)
    try:
        assert not runner.forward(tok, 34, slice(0, 2)).any()
    finally:
        del norm.forward
    handle = torch.nn.modules.module.register_module_forward_hook(
        lambda mod, args, out: calls.append(mod))
    try:
        runner.forward(tok, 34, slice(0, 2))
    finally:
        handle.remove()
    assert sum(mod is norm for mod in calls) == 1
