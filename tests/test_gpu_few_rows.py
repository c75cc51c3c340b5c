"""The few-rows kernel (fewrows_gfx950.hip): one to 64 batch rows, at the edges of its walks (waves without a tile, one,
two and three tiles per wave, odd and even), of its row blocks (ragged for two and four per workgroup) and of its batches, on
pre-sliced codes and on planes."""
import numpy as np
import pytest
import torch

from matgptq_amd import _lib
from oracle import matgptq_oracle as o
from tests import _gpu_util as G

pytestmark = pytest.mark.gpu

# (N, K, M, row blocks per workgroup of 4-bit codes, of 4-bit planes)
CASES = [(16, 128, 1, 1, 1), (48, 1024, 2, 1, 1), (304, 1152, 2, 1, 1), (48, 7680, 4, 1, 1), (5136, 384, 3, 2, 2), (32, 2048, 5, 1, 1),
         (5136, 1152, 8, 2, 2), (8208, 2944, 7, 2, 2), (10256, 3072, 8, 4, 4), (80, 4224, 9, 1, 1), (5136, 896, 16, 2, 2),
         (10256, 1024, 13, 4, 4), (10288, 2176, 16, 4, 4)]
# (N, K, M, row blocks and batch rows per workgroup of 4-bit codes)
MORE_ROWS = [(128, 1024, 64, 1, 16), (2048, 1152, 17, 1, 16), (1360, 2176, 48, 1, 16), (2096, 3200, 31, 2, 16), (4112, 2176, 18, 2, 32),
             (4144, 4096, 32, 2, 32), (8240, 1152, 25, 4, 32), (4128, 512, 48, 2, 16), (16464, 2176, 31, 8, 32), (2080, 1152, 45, 2, 16), (4128, 2176, 41, 4, 16),
             (2064, 2176, 50, 2, 32), (4160, 1152, 64, 4, 32)]
FORMATS = [(2, 128, False), (3, 128, False), (4, 128, False), (6, 128, False), (8, 128, False), (2, -1, True), (3, -1, True),
           (4, 128, True), (6, 128, True), (8, -1, True), (8, 128, True), (4, -1, False)]
# what the operand of bf16 storage carries besides the code (raw_operand.h; planes at 2 bits: 8)
BF16_BASE = {2: 8, 3: 8, 4: 16, 6: 128, 8: 0}


def layer(bits, group, bf16, zeros, n, k, seed):
    dt = torch.bfloat16 if bf16 else torch.float16
    q, s, z = o.make_layer(n, k, group, seed=seed, symmetric=not zeros)
    st, zt = torch.from_numpy(s).to(dt), torch.from_numpy(z).to(dt)
    reorder = lambda t: G.reorder_device(t.view(torch.float16).numpy(), n, k, group)  # (moves 16-bit values, whatever they are)
    return q, st, zt, reorder(st), reorder(zt) if zeros else None


def exact_weights(q, s, z, bits, group):
    """scale * (code - zero) in 64 bits: the kernel multiplies codes as they are and rounds no weight."""
    n, k = q.shape
    spread = lambda t: np.repeat(t.double().numpy(), k if group == -1 else group, axis=1)
    return spread(s) * ((o.slice_codes(q, bits).astype(np.float64) * (1 << (8 - bits))) - spread(z))


def run(bits, group, n, k, x, packed, scales, zeros, flags, planes):
    y = torch.full((x.shape[0], n), float("nan"), dtype=x.dtype, device=G.DEV)
    z = zeros.data_ptr() if zeros is not None else None
    if planes:
        _lib.check(G.lib().matgptq_gemm_master(bits, group, n, k, x.shape[0], packed.data_ptr(), scales.data_ptr(), z, x.data_ptr(),
                                               y.data_ptr(), None, 0, G.stream(), flags))
    else:
        _lib.check(G.lib().matgptq_gemm(bits, group, n, k, x.shape[0], packed.data_ptr(), scales.data_ptr(), z, x.data_ptr(),
                                        y.data_ptr(), G.stream(), flags))
    return y


def packed_of(q, bits, planes):
    if not planes:
        return G.pack_device(q, bits, True)
    n, k = q.shape
    out = torch.empty(G.lib().matgptq_master_words(n, k), dtype=torch.int32, device=G.DEV)
    codes = G.to_dev(q)
    _lib.check(G.lib().matgptq_pack_master_device(codes.data_ptr(), n, k, out.data_ptr(), G.stream()))
    return out


def check(bits, group, bf16, planes, zeros, n, k, m, flags):
    q, st, zt, sd, zd = layer(bits, group, bf16, zeros, n, k, seed=n + k + bits)
    x = torch.from_numpy(o.make_activations(m, k, seed=m, outlier_frac=0.01)).to(st.dtype)
    y = run(bits, group, n, k, x.cuda(), packed_of(q, bits, planes), sd, zd, flags, planes).double().cpu().numpy()
    xd = x.double().numpy()
    ref = xd @ exact_weights(q, st, zt, bits, group).T
    # one rounding of the result, and sums in fp32 whose rounding errors stay below 2^-21 of the sum of the magnitudes: code and
    # zero point around the centre, 2^(b-1) each, on bf16 storage once more twice the base that the operand carries
    scale = np.repeat(st.double().numpy(), k if group == -1 else group, axis=1) * (1 << (8 - bits))
    reach = np.abs(xd) @ (scale * ((1 << bits) + (2 * BF16_BASE[bits] + (1 << bits) if bf16 else 0))).T
    assert np.all(np.abs(y - ref) <= 2.0 ** (-8 if bf16 else -11) * np.abs(ref) + 2.0 ** -21 * reach + 2.0 ** -24)


# (up to four rows of fp16 at group 128, pre-sliced, are the gemv kernel's, as with a fused prologue)
@pytest.mark.parametrize("n,k,m,rows,bits,group,bf16,planes", [
    (n, k, m, min(rows_planes if planes else rows, 4 if bits <= (4 if planes else 6) else 2), bits, group, bf16, planes)
    for n, k, m, rows, rows_planes in CASES for bits, group, bf16 in FORMATS for planes in (False, True)
    if m > 4 or planes or bf16 or group != 128])
def test_few_rows(n, k, m, rows, bits, group, bf16, planes):
    flags = 3 if bf16 else 1
    assert G.lib().matgptq_few_rows(bits, group, n, k, m, flags, int(planes)) == rows
    check(bits, group, bf16, planes, (n // 16 + bits) % 2 == 0, n, k, m, flags)


def rows_expected(k, m, r, rows, bits, group, bf16, planes):
    if not bf16 and group == 128 and m >= 32:
        return 0
    most = 2 if bits > (4 if planes else 6) else 8 if rows == 32 and bits <= 4 and not planes else 4
    small_tiles = planes and bits > 4 and r == 2 and rows == 16 and 1024 < k and m <= 32
    return 0 if small_tiles or r > most else r


@pytest.mark.parametrize("n,k,m,rows,bits,group,bf16,planes", [
    (n, k, m, rows_expected(k, m, r, rows, *form, planes), *form, planes)
    for n, k, m, r, rows in MORE_ROWS for form in FORMATS for planes in (False, True) if rows_expected(k, m, r, rows, *form, planes)])
def test_few_rows_17_to_64(n, k, m, rows, bits, group, bf16, planes):
    flags = 3 if bf16 else 1
    assert G.lib().matgptq_few_rows(bits, group, n, k, m, flags, int(planes)) == rows
    check(bits, group, bf16, planes, (n // 16 + bits) % 2 == 0, n, k, m, flags)


@pytest.mark.parametrize("planes", (False, True))
@pytest.mark.parametrize("bits,group,bf16,zeros", [(4, 128, False, True), (3, -1, False, True), (8, 128, True, False), (6, -1, True, True)])
@pytest.mark.parametrize("n,m", [(80, 11), (80, 28), (4112, 19)])
def test_rows_keep_their_bits_whatever_their_neighbours_hold(n, m, bits, group, bf16, zeros, planes):
    k = 2176
    q, st, _, sd, zd = layer(bits, group, bf16, zeros, n, k, seed=bits)
    packed = packed_of(q, bits, planes)
    x = torch.from_numpy(o.make_activations(m, k, seed=5)).to(st.dtype)
    alone = run(bits, group, n, k, x.cuda(), packed, sd, zd, 3 if bf16 else 1, planes)
    x[3, 300], x[3, 2100], x[8, 7] = float("inf"), float("nan"), float("-inf")
    y = run(bits, group, n, k, x.cuda(), packed, sd, zd, 3 if bf16 else 1, planes)
    others = [i for i in range(m) if i not in (3, 8)]
    assert torch.equal(y[others].view(torch.int16), alone[others].view(torch.int16))
    assert torch.isnan(y[3]).all() and not torch.isfinite(y[8]).all()


@pytest.mark.parametrize("planes", (False, True))
@pytest.mark.parametrize("bits,group,bf16,zeros", [(4, 128, False, True), (3, -1, False, True), (8, 128, True, False), (6, -1, True, True)])
@pytest.mark.parametrize("n,m,row_blocks", [(80, 11, 1), (80, 28, 1), (4112, 19, 2)])
def test_infinities_nan_and_the_largest_numbers(n, m, row_blocks, bits, group, bf16, zeros, planes):
    # one wave's columns hold them: rows with one are what dequantised weights give, the others stay finite
    k = 2176
    q, st, zt, sd, zd = layer(bits, group, bf16, zeros, n, k, seed=bits)
    x = torch.from_numpy(o.make_activations(m, k, seed=5)).to(st.dtype)
    x[1, 300], x[4, 2100], x[5, 7], x[5, 1200] = float("inf"), float("-inf"), float("inf"), float("nan")
    x[7, 640] = 3e38 if bf16 else 65504.0
    w = (o.dequantize_bf16(q, st.float().numpy(), zt.float().numpy(), bits, group) if bf16
         else o.dequantize(q, st.numpy(), zt.numpy(), bits, group)).astype(np.float64)
    with np.errstate(invalid="ignore", over="ignore"):
        sums = x.double().numpy() @ w.T
        reach = np.abs(x.double().numpy()) @ np.abs(w).T
        ref = torch.from_numpy(sums).to(st.dtype).double().numpy()
    y = run(bits, group, n, k, x.cuda(), packed_of(q, bits, planes), sd, zd, 3 if bf16 else 1, planes).double().cpu().numpy()
    assert G.lib().matgptq_few_rows(bits, group, n, k, m, 3 if bf16 else 1, int(planes)) == row_blocks
    for row, col in ((1, 300), (4, 2100), (5, 7)):
        # (a weight the oracle rounds to nothing may be a rounding of scale * (zero - 128) here, and the product infinite)
        some = w[:, col] != 0
        assert np.count_nonzero(some) > 60 and np.array_equal(y[row][some], ref[row][some], equal_nan=True)
    fine = [i for i in range(m) if i not in (1, 4, 5)]
    # (sums that the rounding of the oracle's weights, at most 2^-10 of each product (bf16: 2^-7), can take across the largest
    # number may be either)
    edge = np.abs(np.abs(sums) - torch.finfo(st.dtype).max) <= 2.0 ** (-7 if bf16 else -10) * reach
    assert np.all((np.isfinite(y) == np.isfinite(ref))[fine] | edge[fine])
    for row in fine:
        ok = np.isfinite(ref[row]) & np.isfinite(y[row])
        assert np.max(np.abs(y[row][ok] - ref[row][ok]), initial=0) <= (1e-2 if bf16 else 2e-3) * np.max(np.abs(ref[row][ok]), initial=1e-30)


@pytest.mark.parametrize("planes", (False, True))
@pytest.mark.parametrize("bits,group,bf16", [(b, g, bf16) for b in (2, 3, 4, 6, 8) for g in (128, -1) for bf16 in (False, True)])
@pytest.mark.parametrize("n,k", [(96, 4224), (4112, 2176)])
def test_exact_on_integers(n, k, bits, group, bf16, planes):
    # scales 0 and 1, integer activations: every sum is a whole number below 2^24, and is rounded once
    rng = np.random.default_rng(3)
    dt = torch.bfloat16 if bf16 else torch.float16
    q = rng.integers(0, 256, (n, k), dtype=np.uint8)
    scales = torch.from_numpy(np.round(rng.random((n, 1 if group == -1 else k // 128)))).to(dt)
    sd = G.reorder_device(scales.view(torch.float16).numpy(), n, k, group)
    packed = packed_of(q, bits, planes)
    w = torch.from_numpy(exact_weights(q, scales, torch.full_like(scales, 128), bits, group))
    for m in (5, 8, 16, 27):
        x = torch.from_numpy(np.round(rng.standard_normal((m, k)))).to(dt)
        y = run(bits, group, n, k, x.cuda(), packed, sd, None, 3 if bf16 else 1, planes).cpu()
        assert torch.equal(y, (x.double() @ w.T).to(dt)), m


@pytest.mark.parametrize("planes", (False, True))
@pytest.mark.parametrize("bits,group,bf16", [(4, 128, False), (3, 128, True), (8, -1, False)])
@pytest.mark.parametrize("off", (1, 4, 7))
def test_activations_off_16_bytes(off, bits, group, bf16, planes):
    n, k = 272, 1152
    q, st, _, sd, zd = layer(bits, group, bf16, True, n, k, seed=bits)
    packed, flags = packed_of(q, bits, planes), 3 if bf16 else 1
    op = torch.ops.matgptq_cuda.matmul_matgptq_master if planes else torch.ops.matgptq_cuda.matmul_matgptq_zp
    for m in (1, 3, 6, 8, 16, 24, 64, 300):
        x = torch.from_numpy(o.make_activations(m, k, seed=m)).to(st.dtype).cuda()
        view = torch.cat((x.new_zeros(off), x.reshape(-1)))[off:].view(m, k)
        assert view.data_ptr() % 16 == 2 * off
        call = lambda t: op(t, packed.view(torch.uint32), sd.view(st.dtype), zd.view(st.dtype), n, k, bits, group, flags)
        gemv = run(bits, group, n, k, x, packed, sd, zd, flags | (101 << 8), planes) if m <= 8 else None
        # (up to four rows as they are, in one launch: the gemv kernel, which loads them into registers)
        assert torch.equal(call(view), call(x) if m > 4 else gemv), m
        if m <= 8:  # without the operator's copy: the gemv kernel again
            assert torch.equal(run(bits, group, n, k, view, packed, sd, zd, flags, planes), gemv), m


@pytest.mark.parametrize("planes", (False, True))
@pytest.mark.parametrize("bits,group,bf16", FORMATS)
@pytest.mark.parametrize("m", (11, 28))
def test_a_column_of_outliers_leaves_rows_whose_weight_there_is_zero(m, bits, group, bf16, planes):
    # (products with it are zero: nothing of its size may take part in the sums.  bf16: the base of the operand does, at 2^-21
    # of its magnitude as above, which stays below the rounding of an output)
    n, k, col = 272, 2176, 300
    q, st, _, sd, _ = layer(bits, group, bf16, False, n, k, seed=bits)
    q[:, col] = 128
    x = torch.from_numpy(o.make_activations(m, k, seed=m)).to(st.dtype)
    x[:, col] = 1e4 * x.float().std()
    y = run(bits, group, n, k, x.cuda(), packed_of(q, bits, planes), sd, None, 3 if bf16 else 1, planes).double().cpu().numpy()
    assert G.lib().matgptq_few_rows(bits, group, n, k, m, 3 if bf16 else 1, int(planes)) == 1
    ref = x.double().numpy() @ exact_weights(q, st, torch.full_like(st, 128), bits, group).T
    scale = np.repeat(st.double().numpy(), k if group == -1 else group, axis=1) * (1 << (8 - bits))
    rest = np.abs(x.double().numpy())
    rest[:, col] = 0
    reach = rest @ (scale * (1 << bits)).T
    if bf16:
        reach += np.abs(x.double().numpy()) @ (scale * (2 * BF16_BASE[bits] + (1 << bits))).T
    assert np.all(np.abs(y - ref) <= 2.0 ** (-8 if bf16 else -11) * np.abs(ref) + 2.0 ** -21 * reach + 2.0 ** -24)
