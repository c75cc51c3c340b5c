"""The fused operators of a prompt are the torch operators that they stand for, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _bits(t):
    return t.contiguous().view(torch.int16)


@pytest.mark.parametrize("m,heads,kv,ctx", [(1, 4, 2, 7), (17, 5, 1, 64), (130, 24, 8, 131), (515, 3, 3, 600)])
def test_rope_prompt(m, heads, kv, ctx):
    from matgptq_amd import _glue
    from matgptq_amd.decoder import _rotate

    g = _gen(m)
    qkv = torch.randn(m, (heads + 2 * kv) * 128, device=DEV, generator=g).half()
    qkv[0, :8] = torch.tensor([6e-8, -6e-8, 0.0, -0.0, 65504.0, 1e-4, float("inf"), -1e-7])
    pos = torch.randperm(ctx, device=DEV, generator=g)[:m].contiguous()
    ang = torch.rand(m, 128, device=DEV, generator=g) * 6.28
    cos, sin = ang.cos().half(), ang.sin().half()
    caches = [torch.randn(kv, ctx, 128, device=DEV, generator=g).half() for _ in range(2)]
    want_k, want_v = (c.clone() for c in caches)
    t = qkv.view(m, heads + 2 * kv, 128)
    qk = _rotate(t[:, :heads + kv], cos, sin)
    want_k.index_copy_(1, pos, qk[:, heads:].transpose(0, 1))
    want_v.index_copy_(1, pos, t[:, heads + kv:].transpose(0, 1))
    q_out, before = torch.empty(heads, m, 128, device=DEV, dtype=torch.float16), qkv.clone()
    _glue.rope_prompt(qkv, cos, sin, pos, q_out, *caches, heads, kv)
    assert torch.equal(_bits(q_out), _bits(qk[:, :heads].transpose(0, 1)))
    assert torch.equal(_bits(caches[0]), _bits(want_k)) and torch.equal(_bits(caches[1]), _bits(want_v))
    assert torch.equal(_bits(qkv), _bits(before))
    back = torch.empty(m, heads * 128, device=DEV, dtype=torch.float16)
    _glue.heads_to_rows(q_out, back)
    assert torch.equal(_bits(back), _bits(qk[:, :heads].reshape(m, heads * 128)))


def test_silu_mul_prompt_on_every_gate_value():
    from matgptq_amd import _glue

    gate = torch.arange(-32768, 32768, device=DEV, dtype=torch.int32).to(torch.int16).view(torch.float16).view(64, 1024)
    up = torch.randn(64, 1024, device=DEV, generator=_gen(1)).half()
    up[::2] = 1.0
    out = torch.empty_like(up)
    _glue.silu_mul(torch.cat((gate, up), dim=1), out, prompt=True)
    want = torch.nn.functional.silu(gate) * up
    assert torch.equal(torch.isnan(out), torch.isnan(want))
    assert torch.equal(_bits(torch.nan_to_num(out)), _bits(torch.nan_to_num(want)))


@pytest.mark.parametrize("heads,kv,rows,start,context", [(4, 2, 17, 0, 80), (4, 1, 200, 33, 240), (8, 8, 129, 0, 8300)])
def test_fused_prompt_equals_prompt_of_torch_operators(heads, kv, rows, start, context):
    from matgptq_amd import decoder as D

    cfg = D.DecoderConfig(hidden=heads * 128, ffn=768, layers=2, heads=heads, kv_heads=kv, vocab=512)
    dec = D.random_mixnmatch_decoder(cfg, context, seed=11)[0]
    cache = dec.new_cache()
    if start:
        dec(torch.randint(0, cfg.vocab, (start,), device=DEV, generator=_gen(1)), torch.arange(start, device=DEV), cache)
    tokens = torch.randint(0, cfg.vocab, (rows,), device=DEV, generator=_gen(2))
    pos = torch.arange(start, start + rows, device=DEV)
    cache_a, cache_b = cache.clone(), cache.clone()
    assert dec.fused_prompt_applies(pos, cache_a)
    assert not dec.fused_prompt_applies(pos.int(), cache_a)
    assert not dec.fused_prompt_applies(pos, cache.transpose(0, 1).contiguous().transpose(0, 1))
    a = dec(tokens, pos, cache_a)
    dec.fused = False
    b = dec(tokens, pos, cache_b)
    assert torch.equal(a, b) and torch.equal(_bits(cache_a), _bits(cache_b))


def test_fused_prompt_takes_linears_that_return_views():
    # a linear may be any module: one that hands out part of a larger buffer, off 16 bytes or with longer rows
    from matgptq_amd import decoder as D

    class Part(torch.nn.Module):
        def __init__(self, linear, offset, pad):
            super().__init__()
            self.linear, self.offset, self.pad = linear, offset, pad

        def forward(self, x):
            y = self.linear(x)
            buffer = torch.zeros(self.offset + y.shape[0] * (y.shape[1] + self.pad), dtype=y.dtype, device=y.device)
            part = buffer[self.offset:].view(y.shape[0], -1)[:, :y.shape[1]]
            return part.copy_(y)

    cfg = D.DecoderConfig(hidden=512, ffn=768, layers=2, heads=4, kv_heads=2, vocab=512)
    dec = D.random_mixnmatch_decoder(cfg, 80, seed=3)[0]
    for block, (offset, pad) in zip(dec.blocks, ((4, 0), (8, 24))):
        block.qkv, block.gate_up = Part(block.qkv, offset, pad), Part(block.gate_up, offset, pad)
    tokens, pos = torch.randint(0, cfg.vocab, (33,), device=DEV, generator=_gen(4)), torch.arange(33, device=DEV)
    caches = [dec.new_cache() for _ in range(2)]
    assert dec.fused_prompt_applies(pos, caches[0])
    a = dec(tokens, pos, caches[0])
    dec.fused = False
    b = dec(tokens, pos, caches[1])
    assert torch.equal(a, b) and torch.equal(_bits(caches[0]), _bits(caches[1]))
