"""The fused elementwise kernels of the decode step on the GPU: the rotary embedding with its K/V
writes (bit for bit the eager operations of transformers) and the residual addition with its RMSNorm
(the rule of test_gpu_rmsnorm: equal but where two fp32 sums of squares straddle a rounding)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import bf16_bits
from oracle import numerics as ora

pytestmark = pytest.mark.gpu


def _bf16(gen, *shape):
    return torch.randn(*shape, generator=gen).to(torch.bfloat16)


@pytest.mark.parametrize("h,h_kv,d,nseq,ntok,start,bs", [
    (32, 8, 128, 64, 1, 1024, 16),  # a full decode batch, first slot of a block
    (24, 8, 128, 3, 5, 13, 16),     # a chunk across blocks
    (4, 4, 16, 1, 1, 0, 1),         # the smallest head and block
    (6, 2, 80, 2, 7, 6, 7),         # a head whose units do not fill the last workgroup
])
@pytest.mark.parametrize("stacked", [True, False])
def test_rope_kv(pkg, dev, h, h_kv, d, nseq, ntok, start, bs, stacked):
    from transformers.models.llama.modeling_llama import apply_rotary_pos_emb

    gen = torch.Generator().manual_seed(h * d + start)
    tokens, end = nseq * ntok, start + ntok
    if stacked:  # column views of one stacked product
        qkv = _bf16(gen, tokens, (h + 2 * h_kv) * d).to(dev)
        q, k, v = qkv.split([h * d, h_kv * d, h_kv * d], 1)
    else:
        q, k, v = (_bf16(gen, tokens, n * d).to(dev) for n in (h, h_kv, h_kv))
    angle = torch.rand(tokens, d, generator=gen) * 6.3
    cos, sin = angle.cos().to(torch.bfloat16).to(dev), angle.sin().to(torch.bfloat16).to(dev)
    blocks = -(-end // bs)
    table = torch.randperm(nseq * blocks, generator=gen).reshape(nseq, blocks).to(torch.int32).to(dev)
    cache = [_bf16(gen, nseq, h_kv, end + 3, d).to(dev) for _ in range(2)]
    pool = [_bf16(gen, nseq * blocks + 1, bs, h_kv, d).to(dev) for _ in range(2)]
    want_cache, want_pool = [t.clone() for t in cache], [t.clone() for t in pool]

    split = lambda t, n: t.reshape(nseq, ntok, n, d).transpose(1, 2)  # noqa: E731
    rq, rk = apply_rotary_pos_emb(split(q, h), split(k, h_kv), cos.reshape(nseq, ntok, d),
                                  sin.reshape(nseq, ntok, d))
    pos = torch.arange(start, end, device=dev)
    where = table[:, pos // bs].long()
    for t, p, new in zip(want_cache, want_pool, (rk, split(v, h_kv))):
        t[:, :, start:end] = new
        p[where, (pos % bs).expand_as(where)] = new.transpose(1, 2)

    got = pkg.ops.rope_kv(q, k, v, cos, sin, h, h_kv, nseq, start, tuple(cache), (*pool, table))
    assert torch.equal(got, rq.transpose(1, 2).reshape(tokens, h, d))
    for a, b in zip(cache + pool, want_cache + want_pool):
        assert torch.equal(a, b)
    # Without a cache or pool only q comes back.
    assert torch.equal(pkg.ops.rope_kv(q, k, v, cos, sin, h, h_kv, nseq, start), got)


@pytest.mark.parametrize("m,k", [(1, 8), (64, 4096), (3, 4104), (5, 3072), (2, 8192), (2, 16384)])
@pytest.mark.parametrize("residual", [True, False])
def test_add_rmsnorm(pkg, dev, m, k, residual):
    gen = torch.Generator().manual_seed(m + k)
    x, r = _bf16(gen, m, k).to(dev), _bf16(gen, m, k).to(dev)
    w = (1 + 0.1 * torch.randn(k, generator=gen)).to(torch.bfloat16).to(dev)
    s, y = pkg.ops.add_rmsnorm(x, r if residual else None, w, 1e-5)
    want = x + r if residual else x
    assert torch.equal(s, want)
    ref = ora.rmsnorm_bf16(bf16_bits(want), bf16_bits(w), 1e-5)
    ulps = ora.bf16_ulps_apart(bf16_bits(y), ora.bf16_bits_to_f32(ref).astype(np.float64))
    assert ulps.max() <= 2 and np.mean(ulps > 0) < 1e-3 + 1.0 / ulps.size


@pytest.mark.parametrize("m,k", [(1, 8), (5, 4104), (3, 16384)])
@pytest.mark.parametrize("into", ["x", "res"])
def test_add_rmsnorm_in_place(pkg, dev, m, k, into):
    """The sum written over one of its operands, as the C entry allows."""
    gen = torch.Generator().manual_seed(m * k)
    x, r = _bf16(gen, m, k).to(dev), _bf16(gen, m, k).to(dev)
    w = (1 + 0.1 * torch.randn(k, generator=gen)).to(torch.bfloat16).to(dev)
    s, y = pkg.ops.add_rmsnorm(x, r, w, 1e-5)
    got = torch.empty_like(y)
    target = x if into == "x" else r
    status = pkg.library().lse_add_rmsnorm(
        x.data_ptr(), k, r.data_ptr(), k, w.data_ptr(), 1e-5, target.data_ptr(), got.data_ptr(), m,
        k, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert status == 0 and torch.equal(target, s) and torch.equal(got, y)


def test_add_rmsnorm_takes_a_piece_of_a_flat_weight(pkg, dev):
    """A contiguous weight at an address no 16-byte load takes: the same result as its aligned copy."""
    gen = torch.Generator().manual_seed(5)
    x, flat = _bf16(gen, 3, 64).to(dev), _bf16(gen, 65).to(dev)
    want = pkg.ops.add_rmsnorm(x, None, flat[1:].clone(), 1e-5)[1]
    assert torch.equal(pkg.ops.add_rmsnorm(x, None, flat[1:], 1e-5)[1], want)


def test_rejections(pkg, dev):
    x = torch.zeros(2, 16392, dtype=torch.bfloat16, device=dev)
    with pytest.raises(RuntimeError, match="range"):
        pkg.ops.add_rmsnorm(x, None, x[0].contiguous(), 1e-5)
    z = torch.zeros(2, 32, dtype=torch.bfloat16, device=dev)
    cache = torch.zeros(2, 2, 4, 16, dtype=torch.bfloat16, device=dev)
    with pytest.raises(RuntimeError, match="cache"):
        pkg.ops.rope_kv(z, z, z, z[:, :16], z[:, :16], 2, 2, 2, 4, (cache, cache))
    table = torch.zeros(2, 1, dtype=torch.int32, device=dev)
    with pytest.raises(RuntimeError, match="table"):
        pkg.ops.rope_kv(z, z, z, z[:, :16], z[:, :16], 2, 2, 2, 4, None,
                        (cache.transpose(1, 2), cache.transpose(1, 2), table))
