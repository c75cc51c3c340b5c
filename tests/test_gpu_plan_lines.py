"""Formats and sizes on the lines of the rules that choose between 128 x 128 tiles, 128 x 192 tiles (with K split, alone, or mixed
with the narrower ones in one launch), 64 x 128 tiles and the mid-batch kernel, against the product in 64 bits and against the
128 x 128 tile forced."""
import numpy as np
import pytest
import torch

from matgptq_amd import _lib
from oracle import matgptq_oracle as o
from tests import _gpu_util as G
from tests.test_gpu_few_rows import layer, packed_of, run

pytestmark = pytest.mark.gpu

# (bits, group, bf16, zeros, N, K, M, plan)
CASES = [(6, -1, False, False, 5984, 2176, 1000, "cfg13"), (3, 128, True, True, 5984, 2176, 1000, "cfg13"),
         (8, 32, True, True, 6096, 2176, 1024, "cfg13"), (2, 32, False, True, 5984, 2176, 1000, "cfg13"),
         (6, 128, True, True, 10240, 256, 1024, "cfg14"), (6, -1, False, False, 10240, 256, 1000, "cfg14"),
         (8, 32, True, True, 10256, 256, 1000, "cfg9"), (6, 32, True, True, 12288, 256, 1024, "cfg9"),
         (3, 32, True, True, 10256, 256, 1000, "cfg3"), (6, 128, False, True, 5984, 2176, 1000, "cfg3"),
         (6, 128, False, False, 10240, 256, 1024, "cfg9"),
         (4, 32, False, True, 4608, 2176, 121, "R2 mb2"), (2, 128, True, False, 3072, 2176, 192, "R4 mb4"),
         (8, -1, False, True, 1552, 3200, 130, "R2 mb2"), (4, -1, False, True, 1552, 2176, 641, "cfg16")]


@pytest.mark.parametrize("bits,group,bf16,zeros,n,k,m,plan", CASES)
def test_plan_lines(bits, group, bf16, zeros, n, k, m, plan):
    flags = 3 if bf16 else 1
    assert _lib.describe_plan(bits, group, n, k, m, zeros, flags).endswith(plan)
    q, st, zt, sd, zd = layer(bits, group, bf16, zeros, n, k, seed=n + bits)
    x = torch.from_numpy(o.make_activations(m, k, seed=m)).to(st.dtype).cuda()
    packed = packed_of(q, bits, False)
    y = run(bits, group, n, k, x, packed, sd, zd, flags, False).double()
    ref = run(bits, group, n, k, x, packed, sd, zd, flags | ((64 + 3) << 8), False).double()
    # both form the same rounded weights and round each result once; their sums in fp32, in other orders, differ by less than
    # 2^-20 of the sum of the magnitudes
    spread = lambda t: np.repeat(t.double().numpy(), k if group == -1 else group, axis=1)
    w = torch.from_numpy(spread(st) * (o.slice_codes(q, bits).astype(np.float64) * (1 << (8 - bits)) - spread(zt))).cuda()
    reach = x.double().abs() @ w.abs().T
    # against weights that are not rounded: half a step of each weight besides, and (fp16 storage) of scale times zero point
    shift = torch.from_numpy(spread(st) * np.abs(spread(zt) - 128.0)).cuda()
    half = 2.0 ** (-8 if bf16 else -11)
    weights = half * reach if bf16 else half * (reach + x.double().abs() @ shift.T)
    exact = x.double() @ w.T
    assert torch.all((y - exact).abs() <= half * exact.abs() + weights + 2.0 ** -20 * reach + 2.0 ** -24)
    assert torch.all((y - ref).abs() <= 2.0 ** (-7 if bf16 else -10) * ref.abs() + 2.0 ** -20 * reach + 2.0 ** -24)
