"""The one-launch packing of a layer (codes, scales, zeros) against the separate host packers, word for
word, at the edges of its tiling: a workgroup takes eight tiles of K, half a wave one tile."""
import numpy as np
import pytest
import torch

import matgptq_cuda  # noqa: F401  (registers the operators)
from matgptq_amd import _lib
from oracle import matgptq_oracle as o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("source", (0, 1, 2))
@pytest.mark.parametrize("b", (2, 3, 4, 6, 8))
@pytest.mark.parametrize("n,k,g", ((16, 128, 128), (48, 7 * 128, 32), (32, 8 * 128, -1), (80, 9 * 128, 128),
                                   (32, 8 * 128 + 64, 32), (16, 192, -1), (48, 17 * 128 + 64, 32)))
def test_layer_in_one_launch_equals_host_packers(n, k, g, b, source):
    if source == 2 and k % 128 != 0:
        pytest.skip("the planes have whole tiles only")
    L = _lib.load()
    rng = np.random.default_rng(n + k + b)
    q = rng.integers(0, 256, (n, k), dtype=np.uint8)
    codes = o.slice_codes(q, b) if source == 0 else q
    groups = 1 if g == -1 else k // g
    per_group = [rng.integers(0, 1 << 16, (n, groups), dtype=np.uint16) for _ in range(2)]
    dev = [torch.from_numpy(t.view(np.float16)).cuda() for t in per_group]
    packed, scales, zeros = torch.ops.matgptq_cuda.pack_matgptq_layer(
        torch.from_numpy(codes).cuda(), dev[0], dev[1], b, g, source)
    if source == 2:
        host = np.zeros(L.matgptq_master_words(n, k), dtype=np.uint32)
        _lib.check(L.matgptq_pack_master_host(q.ctypes.data, n, k, host.ctypes.data))
    else:
        host = np.zeros(L.matgptq_packed_words(b, n, k), dtype=np.uint32)
        _lib.check(L.matgptq_pack_host(q.ctypes.data, n, k, b, 1, host.ctypes.data))
    assert np.array_equal(packed.cpu().numpy(), host)
    for got, src in ((scales, per_group[0]), (zeros, per_group[1])):
        want = np.zeros_like(src)
        _lib.check(L.matgptq_reorder_scales_host(src.ctypes.data, n, k, g, want.ctypes.data))
        assert np.array_equal(got.cpu().numpy().view(np.uint16), want)
    without = torch.ops.matgptq_cuda.pack_matgptq_layer(torch.from_numpy(codes).cuda(), dev[0], None, b, g, source)
    assert len(without) == 2 and torch.equal(without[0].view(torch.int32), packed.view(torch.int32))


@pytest.mark.parametrize("b", (2, 3, 4, 6, 8))
@pytest.mark.parametrize("offset", (0, 1, 4, 8, 12, 16))
@pytest.mark.parametrize("count", (1, 15, 16, 63, 4096 * 16 + 7))
def test_slice_at_every_alignment(count, offset, b):
    # 16 bytes per thread where the codes lie on 4 bytes, code by code elsewhere and at the end
    L = _lib.load()
    q = np.random.default_rng(count + offset).integers(0, 256, count, dtype=np.uint8)
    src = torch.zeros(count + offset, dtype=torch.uint8, device="cuda")
    src[offset:] = torch.from_numpy(q).cuda()
    for out_offset in {0, offset}:
        out = torch.full((count + out_offset + 16,), 255, dtype=torch.uint8, device="cuda")
        _lib.check(L.matgptq_slice_device(src.data_ptr() + offset, count, b, out.data_ptr() + out_offset,
                                          torch.cuda.current_stream().cuda_stream))
        got = out.cpu().numpy()
        assert np.array_equal(got[out_offset:out_offset + count], o.slice_codes(q, b))
        assert (got[:out_offset] == 255).all() and (got[out_offset + count:] == 255).all()


def test_layer_on_the_gpu_is_refused_in_the_words_of_the_separate_packers():
    from matgptq_cuda.matgptq_linear import MatGPTQLinear

    q = torch.zeros(32, 256, dtype=torch.uint8, device="cuda")
    s = torch.ones(32, 2, dtype=torch.float16, device="cuda")
    for codes, scales, message in ((torch.zeros(256, 32, dtype=torch.uint8, device="cuda").t(), s, "qweights must be contiguous"),
                                   (q.int(), s, "qweights must be uint8"),
                                   (q, torch.ones(2, 32, dtype=torch.float16, device="cuda").t(), "scales must be contiguous"),
                                   (q, s.float(), "scales must be float16 or bfloat16"),
                                   (q, s[:16].contiguous(), "scales must have shape")):
        with pytest.raises(RuntimeError, match=message):
            MatGPTQLinear(codes, scales, 4, 128)
