"""What the decoder decides on the host, with blocks that only note what they are given."""
import pytest
import torch

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
