"""What the decoder decides on the host, with blocks that only note what they are given."""
import pytest
import torch
from torch._subclasses import FakeTensor, FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx
from torch.utils._python_dispatch import TorchDispatchMode

from matgptq_amd import _glue
from matgptq_amd import decoder as D


class _Block(torch.nn.Module):
    def __init__(self):
        super().__init__()
        self.workspaces = []

    def forward_fused(self, h, delta, x, cos, sin, pos, k_cache, v_cache, attn_workspace):
        self.workspaces.append(attn_workspace)
        return torch.zeros_like(h)


def _decoder(monkeypatch, context, heads=4, kv_heads=2):
    monkeypatch.setattr(_glue, "add_rmsnorm", lambda h, delta, weight, x, eps: x.copy_(h))
    cfg = D.DecoderConfig(hidden=heads * 128, ffn=256, layers=2, heads=heads, kv_heads=kv_heads, vocab=16)
    embed = torch.zeros(cfg.vocab, cfg.hidden, dtype=torch.float16)
    return D.Decoder(cfg, [_Block(), _Block()], embed, embed.clone(), context)


def _step(decoder, rows):
    cache = torch.zeros(2, 2, decoder.cfg.kv_heads, decoder.max_context, 128, dtype=torch.float16)
    decoder(torch.zeros(rows, dtype=torch.int64), torch.arange(rows), cache)
    return [block.workspaces[-1] for block in decoder.blocks]


@pytest.mark.parametrize("rows", (1, 2, 8, 16))
def test_steps_do_not_share_their_attention_workspace(monkeypatch, rows):
    # two sessions of one decoder on two streams: a shared workspace would mix their partial results
    decoder = _decoder(monkeypatch, context=1100)
    first, second = _step(decoder, rows), _step(decoder, rows)
    assert first[0] is first[1] and second[0] is second[1]  # the blocks of a step follow one another
    assert first[0].data_ptr() != second[0].data_ptr()
    for workspace in (first[0], second[0]):
        assert workspace.numel() >= _glue.load().matgptq_glue_attention_workspace_floats(rows, 4, 1100)


@pytest.mark.parametrize("context", (64, 1100))
def test_split_attention_switches_the_split_for_every_number_of_rows(monkeypatch, context):
    decoder = _decoder(monkeypatch, context)
    assert decoder.split_attention == (context > 768)
    assert (_step(decoder, 8)[0] is not None) == (context > 768) and _step(decoder, 1)[0] is not None
    for on in (False, True):
        decoder.split_attention = on
        assert [(_step(decoder, rows)[0] is not None) for rows in (1, 8)] == [on, on]


def test_ratios_that_the_split_does_not_cover(monkeypatch):
    decoder = _decoder(monkeypatch, 1100, heads=6, kv_heads=2)
    assert not decoder.split_attention and _step(decoder, 1)[0] is None and _step(decoder, 8)[0] is None


class _Dense(torch.nn.Module):
    def __init__(self, n, k, device):
        super().__init__()
        self.w = torch.nn.Parameter(torch.zeros(n, k, dtype=torch.float16, device=device), requires_grad=False)

    def forward(self, x):
        return torch.nn.functional.linear(x, self.w)


def _dense_decoder(device, context=64):
    cfg = D.DecoderConfig(hidden=512, ffn=256, layers=2, heads=4, kv_heads=2, vocab=16)
    blocks = [D.Block(cfg, {name: _Dense(*shape, device) for name, shape in cfg.linear_shapes().items()}, torch.float16,
                      device) for _ in range(cfg.layers)]
    embed = torch.zeros(cfg.vocab, cfg.hidden, dtype=torch.float16, device=device)
    return D.Decoder(cfg, blocks, embed, embed.clone(), context)


def test_prompt_of_fake_tensors_runs_on_torch_operators():
    # shapes worked out without memory, as exporters and compilers do: there is nothing to hand to a kernel
    with FakeTensorMode():
        decoder = _dense_decoder("cuda")
        cache = decoder.new_cache()
        logits = decoder(torch.zeros(20, dtype=torch.int64, device="cuda"), torch.arange(20, device="cuda"), cache)
        assert logits.shape == (1, 16) and not decoder.fused_prompt_applies(torch.arange(20, device="cuda"), cache)


def test_plain_tensors_are_not_traced_transformed_or_watched():
    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    seen = []

    def look(t):
        seen.append(D._plain_tensors(t))
        return t + 1

    x = torch.zeros(3)
    look(x)
    assert seen == [True]
    torch.func.vmap(look)(x)
    torch.jit.trace(look, x, check_trace=False)
    make_fx(look)(x)
    torch.export.export(_Look(look), (x,), strict=False)
    with Watch():
        look(x)
    with FakeTensorMode() as mode:
        look(mode.from_tensor(x))
    assert len(seen) >= 7 and not any(seen[1:])


class _Look(torch.nn.Module):
    def __init__(self, look):
        super().__init__()
        self.look = look

    def forward(self, x):
        return self.look(x)


def test_replaced_block_forward_gets_the_arguments_of_a_block(monkeypatch):
    # a block whose forward was replaced on the instance, or that was compiled, is called as a block always was
    monkeypatch.setattr(D, "_plain_tensors", lambda *_: True)
    with FakeTensorMode():
        decoder = _dense_decoder("cuda")
        cache, pos = decoder.new_cache(), torch.arange(20, device="cuda")
        monkeypatch.setattr(FakeTensor, "data_ptr", lambda self: 4096, raising=False)
        assert decoder.fused_prompt_applies(pos, cache)
        original = decoder.blocks[1].forward
        decoder.blocks[1].forward = lambda h, cos, sin, pos, k_cache, v_cache, bias: original(h, cos, sin, pos, k_cache,
                                                                                              v_cache, bias)
        assert not decoder.fused_prompt_applies(pos, cache)
        assert decoder(torch.zeros(20, dtype=torch.int64, device="cuda"), pos, cache).shape == (1, 16)
        del decoder.blocks[1].forward
        assert decoder.fused_prompt_applies(pos, cache)
        decoder.blocks[0]._compiled_call_impl = decoder.blocks[0]._call_impl
        assert not decoder.fused_prompt_applies(pos, cache)
