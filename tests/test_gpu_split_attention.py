"""The split attention with one and with two query heads per workgroup (one up to four rows on caches of up to 1024
rows, two elsewhere; glue_gfx950.hip) against 64-bit attention: several workgroups per key/value head, several used
splits, the ends of splits, both sides of the rule."""
import pytest
import torch

from matgptq_amd import _glue

pytestmark = pytest.mark.gpu

DEV, D = "cuda", 128


def _inputs(m, heads, kv, ctx, positions):
    g = torch.Generator(device=DEV).manual_seed(ctx + 7 * m + heads)
    qkv = torch.randn(m, (heads + 2 * kv) * D, device=DEV, generator=g).half()
    caches = [torch.randn(kv, ctx, D, device=DEV, generator=g).half() for _ in range(2)]
    for c in caches:  # rows that no query may see: read, never used
        c[:, max(positions) + 1:] = float("nan")
    return g, qkv, caches, torch.tensor(positions, device=DEV)


def _check(out, q, k, v, positions, heads, kv):
    """out [m, heads * D] against 64 bits.  Bound: the rounding of the result, and fp32 sums and exponentials over the
    rows in use (2^-14 of the largest value, the error of 1000 additions in fp32)."""
    for i, p in enumerate(positions):
        qi = q[i].double().view(kv, heads // kv, D)
        scores = torch.matmul(qi, k[:, :p + 1].double().transpose(1, 2).contiguous()) * D ** -0.5
        want = torch.matmul(torch.softmax(scores, dim=-1), v[:, :p + 1].double()).view(-1)
        bound = 2.0 ** -11 * want.abs() + 2.0 ** -14 * float(v[:, :p + 1].abs().max())
        assert bool(((out[i].double() - want).abs() <= bound).all()), (i, p)


@pytest.mark.parametrize("heads,kv,ctx,position", [
    (32, 8, 1100, 1099), (64, 8, 2000, 1024), (8, 1, 1500, 64), (4, 2, 1025, 127), (4, 2, 1025, 128), (16, 8, 8192, 5),
    (32, 8, 1024, 1023), (32, 8, 1025, 1024), (64, 8, 1024, 0), (8, 8, 1100, 1050), (64, 8, 4160, 4159)])
def test_one_row_with_rotary(heads, kv, ctx, position):
    g, qkv, (k, v), pos = _inputs(1, heads, kv, ctx, [position])
    ang = torch.rand(ctx, D, device=DEV, generator=g) * 6.28
    cos, sin = ang.cos().half(), ang.sin().half()
    rotated, k_want, v_want = qkv.clone(), k.clone(), v.clone()
    _glue.rope_cache(rotated, cos, sin, pos, k_want, v_want, heads, kv)
    before = qkv.clone()
    for _ in range(2):  # (the second time the row is in the caches already)
        workspace = _glue.attention_workspace(1, heads, ctx, DEV).fill_(float("nan"))
        out = torch.full((1, heads * D), float("nan"), device=DEV, dtype=torch.float16)
        _glue.attention_split(qkv, cos, sin, pos, k, v, out, workspace, heads, kv, fuse_rotary=True)
        _check(out, rotated[:, :heads * D], k_want, v_want, [position], heads, kv)
        # the rows in use and the untouched NaN behind them, bit for bit: one rotary expression in every kernel
        for got, want in ((k, k_want), (v, v_want), (qkv, before)):
            assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("m,heads,kv,ctx,positions", [
    (5, 16, 8, 1100, [0, 63, 64, 700, 1099]), (8, 32, 8, 1300, [5, 127, 128, 129, 640, 1023, 1024, 1299]),
    (16, 8, 1, 2100, [131 * i for i in range(16)]), (4, 32, 8, 1024, [0, 64, 500, 1023]), (4, 32, 8, 1025, [0, 64, 500, 1024]),
    (5, 32, 8, 1024, [1, 64, 191, 500, 1023]), (6, 12, 12, 900, [0, 1, 62, 63, 64, 899]), (2, 64, 8, 5000, [4999, 64])])
def test_several_rows(m, heads, kv, ctx, positions):
    _, qkv, (k, v), pos = _inputs(m, heads, kv, ctx, positions)
    k_before, v_before = k.clone(), v.clone()
    workspace = _glue.attention_workspace(m, heads, ctx, DEV).fill_(float("nan"))
    out = torch.full((m, heads * D), float("nan"), device=DEV, dtype=torch.float16)
    _glue.attention_split(qkv, None, None, pos, k, v, out, workspace, heads, kv, fuse_rotary=False)
    _check(out, qkv[:, :heads * D], k, v, positions, heads, kv)
    assert torch.equal(k.view(torch.int16), k_before.view(torch.int16))
    assert torch.equal(v.view(torch.int16), v_before.view(torch.int16))
