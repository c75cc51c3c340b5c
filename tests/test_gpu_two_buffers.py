"""The mid-batch kernel's walks (skinny_gfx950.hip) at the edges of their ranges: one tile with one buffer and one register
set; two, three and an odd number of tiles with two activation buffers; waves without a tile, more workgroups than CUs, ragged
batches; pre-sliced codes, and walks of one tile on planes."""
import numpy as np
import pytest
import torch

from matgptq_amd import _lib
from oracle import matgptq_oracle as o
from tests import _gpu_util as G
from tests.test_gpu_few_rows import packed_of, run

pytestmark = pytest.mark.gpu

# (N, K, M, forced variant: 80 + {0: one, 1: two, 2: four row blocks} + 3 * {0: 16, 1: 32, 2: 64 batch rows}, formats with two
# buffers: "all", "none", "plain" (not 6 bits, not zero points at group 32), "fp16")
CASES = [(32, 128, 9, 80, "none"), (64, 384, 16, 80, "none"), (48, 1024, 17, 83, "none"), (96, 1024, 16, 81, "none"),
         (160, 896, 40, 85, "none"), (112, 1024, 23, 84, "none"), (208, 1024, 70, 88, "none"), (48, 1152, 33, 83, "all"), (64, 2048, 12, 80, "all"),
         (32, 3072, 16, 80, "all"), (80, 2944, 20, 83, "all"), (32, 3200, 16, 80, "plain"), (48, 8192, 9, 80, "plain"),
         (32, 4992, 31, 83, "fp16"), (8256, 2176, 16, 81, "fp16"), (16640, 1280, 7, 82, "fp16")]
FORMATS = [(4, 128, False), (3, 128, True), (8, 128, False), (2, -1, False), (6, 32, True), (8, 32, False), (8, 32, True)]


def _expected(which, n, variant, bits, group, bf16, zeros):
    if which == "none":
        return False
    if which == "plain":
        return bits != 6 and not (group == 32 and zeros)
    if which == "fp16":
        return not bf16 and not (n > 8000 and bits == 8 and group == 32)
    return True


@pytest.mark.parametrize("zeros", (True, False))
@pytest.mark.parametrize("bits,group,bf16", FORMATS)
@pytest.mark.parametrize("n,k,m,variant,which", CASES)
def test_two_buffers(n, k, m, variant, which, bits, group, bf16, zeros):
    flags = 1 | (2 if bf16 else 0) | (variant << 8)
    buffers = _lib.load().matgptq_midbatch_buffers(bits, group, n, k, m, int(zeros), flags)
    assert buffers == (2 if _expected(which, n, variant, bits, group, bf16, zeros) else 1)
    q, s, z = o.make_layer(n, k, group, seed=n + k + bits, symmetric=not zeros)
    dt = torch.bfloat16 if bf16 else torch.float16
    st, zt = torch.from_numpy(s).to(dt), torch.from_numpy(z).to(dt)
    x = torch.from_numpy(o.make_activations(m, k, seed=m)).to(dt)
    bits_of = lambda t: t.view(torch.float16).numpy()  # (the reordering moves 16-bit values, whatever they are)
    sd, zd = G.reorder_device(bits_of(st), n, k, group), G.reorder_device(bits_of(zt), n, k, group) if zeros else None
    y = G.gemm(bits, group, n, k, x.cuda(), G.pack_device(q, bits, True), sd, zd, flags=flags).view(dt)
    if which == "none":  # the same codes in the same order: the same bits from planes
        ym = run(bits, group, n, k, x.cuda(), packed_of(q, bits, True), sd, zd, flags, True)
        assert torch.equal(y.view(torch.int16), ym.view(torch.int16))
    if bf16:  # the weights are the oracle's; one rounding of the result (half a step of 2^-7), sums in fp32 (a hundredth of it)
        w = o.dequantize_bf16(q, st.float().numpy(), zt.float().numpy(), bits, group)
        ref = x.double().numpy() @ w.astype(np.float64).T
        assert np.max(np.abs(y.double().cpu().numpy() - ref)) <= 1.01 * 2.0 ** -8 * np.max(np.abs(ref))
    else:
        G.assert_close_to_oracle(y.cpu().numpy(), x.numpy(), o.dequantize(q, s, z, bits, group),
                                 f"{n}x{k} m{m} b{bits} g{group} v{variant}")
