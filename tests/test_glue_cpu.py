"""The library of decode-time operators between the linears loads without a GPU, exports what its
header declares, and rejects bad arguments before anything is launched."""
import ctypes
import os
import re

import pytest
import torch

from matgptq_amd import _glue

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_declared_symbol_is_exported():
    header = open(os.path.join(ROOT, "include", "matgptq_glue.h")).read()
    header = re.sub(r"/\*.*?\*/", "", header, flags=re.S)
    names = set(re.findall(r"\b(matgptq_glue_[a-z_0-9]+)\s*\(", header))
    assert names == set(_glue.EXPORTS)
    lib = ctypes.CDLL(_glue.GLUE_PATH)
    for n in sorted(names):
        assert hasattr(lib, n), n
    limit = int(re.search(r"#define MATGPTQ_GLUE_MAX_CONTEXT (\d+)", header).group(1))
    assert limit == _glue.MAX_CONTEXT


def test_argument_checks_come_before_any_launch():
    L = _glue.load()
    one = ctypes.c_void_p(16)  # never dereferenced: every call below fails its checks first
    assert L.matgptq_glue_add_rmsnorm(None, None, one, one, 1, 256, 1e-5, None) == -4
    assert L.matgptq_glue_add_rmsnorm(one, None, one, one, 1, 260, 1e-5, None) == -3
    assert L.matgptq_glue_add_rmsnorm(one, None, one, one, 1, 16384, 1e-5, None) == -8
    assert L.matgptq_glue_rope_cache(one, one, one, None, one, one, 1, 4, 2, 128, 64, None) == -4
    assert L.matgptq_glue_rope_cache(one, one, one, one, one, one, 1, 4, 3, 128, 64, None) == -3
    assert L.matgptq_glue_attention(one, one, one, one, one, 1, 4, 2, 64, 64, None) == -3
    assert L.matgptq_glue_attention(one, one, one, one, one, 1, 4, 2, 128, _glue.MAX_CONTEXT + 1, None) == -8
    assert L.matgptq_glue_rope_attention(one, one, one, one, one, one, None, 4, 2, 128, 64, None) == -4
    assert L.matgptq_glue_rope_attention(one, one, one, one, one, one, one, 4, 2, 64, 64, None) == -3
    assert L.matgptq_glue_attention_split(one, None, None, one, one, one, one, None, 1, 4, 2, 128, 64, 0, None) == -4
    assert L.matgptq_glue_attention_split(one, None, None, one, one, one, one, one, 1, 4, 2, 128, 64, 1, None) == -4
    assert L.matgptq_glue_attention_split(one, one, one, one, one, one, one, one, 2, 4, 2, 128, 64, 1, None) == -3
    assert L.matgptq_glue_attention_split(one, None, None, one, one, one, one, one, 1, 6, 2, 128, 64, 0, None) == -3
    assert L.matgptq_glue_attention_workspace_floats(2, 4, 65) == 2 * 4 * 2 * 130
    assert L.matgptq_glue_argmax(None, one, 1, 8, None) == -4
    assert L.matgptq_glue_argmax(one, one, 0, 8, None) == -3
    assert L.matgptq_glue_argmax(one, one, 1, 2 ** 31, None) == -8
    assert L.matgptq_glue_silu_mul(one, None, 1, 64, None) == -4
    assert L.matgptq_glue_silu_mul(one, one, 1, 60, None) == -3
    assert b"NULL" in L.matgptq_glue_strerror(-4)


class _GpuTensor:
    """What the operators look at in a GPU tensor, without a GPU."""

    is_cuda = True

    def __init__(self, shape, dtype, device):
        self.shape, self.dtype, self.device = torch.Size(shape), dtype, torch.device(device)

    def is_contiguous(self):
        return True

    def dim(self):
        return len(self.shape)

    def numel(self):
        return self.shape.numel()

    def data_ptr(self):
        return 4096

    def get_device(self):
        return self.device.index


class _Gpus:
    """A library whose calls return 0 and note the GPU that was current and the stream they were given; the
    stream of GPU i is 100 + i."""

    def __init__(self, monkeypatch, current=0):
        self.current, self.calls = current, []
        gpus = self

        class Device:
            def __init__(self, device):
                self.index = device

            def __enter__(self):
                self.before, gpus.current = gpus.current, self.index

            def __exit__(self, *_):
                gpus.current = self.before

        class Library:
            def __getattr__(self, name):
                if name == "matgptq_glue_attention_workspace_floats":
                    return lambda rows, heads, ctx: rows * heads * -(-ctx // 64) * 130

                def call(*args):
                    gpus.calls.append((name, gpus.current, args))
                    return 0
                return call

        library = Library()
        monkeypatch.setattr(_glue, "load", lambda: library)
        monkeypatch.setattr(torch.cuda, "device", Device)
        monkeypatch.setattr(torch.cuda, "current_device", lambda: gpus.current)
        monkeypatch.setattr(_glue, "raw_stream", lambda index: 100 + index)


def _operator_calls(device, other=None):
    """(name, call) for every operator on tensors of `device`; with `other` the last tensor is on that one."""
    heads, kv, d, ctx = 4, 2, 128, 96

    def f16(*shape, last=False):
        return _GpuTensor(shape, torch.float16, other if last and other else device)

    def pos(m):
        return _GpuTensor((m,), torch.int64, device)

    def qkv(m):
        return f16(m, (heads + 2 * kv) * d)

    def cache(last=False):
        return f16(kv, ctx, d, last=last)

    def workspace(m):
        return _GpuTensor((m * heads * 2 * 130,), torch.float32, other or device)

    last = other is not None
    return [
        ("add_rmsnorm", lambda: _glue.add_rmsnorm(f16(3, 64), None, f16(64), f16(3, 64, last=last), 1e-5)),
        ("rope_cache", lambda: _glue.rope_cache(qkv(2), f16(ctx, d), f16(ctx, d), pos(2), cache(), cache(last), heads, kv)),
        ("attention", lambda: _glue.attention(qkv(2), cache(), cache(), pos(2), f16(2, heads * d, last=last), heads, kv)),
        ("rope_attention", lambda: _glue.rope_attention(qkv(1), f16(ctx, d), f16(ctx, d), pos(1), cache(), cache(),
                                                        f16(1, heads * d, last=last), heads, kv)),
        ("attention_split", lambda: _glue.attention_split(qkv(2), None, None, pos(2), cache(), cache(), f16(2, heads * d),
                                                          workspace(2), heads, kv, False)),
        ("attention_split", lambda: _glue.attention_split(qkv(1), f16(ctx, d), f16(ctx, d), pos(1), cache(), cache(),
                                                          f16(1, heads * d), workspace(1), heads, kv, True)),
        ("rope_prompt", lambda: _glue.rope_prompt(qkv(5), f16(5, d), f16(5, d), pos(5), f16(heads, 5, d), cache(), cache(last),
                                                  heads, kv)),
        ("heads_to_rows", lambda: _glue.heads_to_rows(f16(heads, 5, d), f16(5, heads * d, last=last))),
        ("silu_mul", lambda: _glue.silu_mul(f16(2, 128), f16(2, 64, last=last))),
        ("silu_mul_prompt", lambda: _glue.silu_mul(f16(2, 128), f16(2, 64, last=last), prompt=True)),
        ("argmax", lambda: _glue.argmax(_GpuTensor((2, 9), torch.float32, device),
                                        _GpuTensor((2,), torch.int64, other or device))),
    ]


def test_every_operator_launches_on_the_gpu_of_its_tensors(monkeypatch):
    # with another GPU current: a launch there would get pointers of the wrong GPU and the wrong GPU's stream
    gpus = _Gpus(monkeypatch, current=0)
    for device in ("cuda:1", "cuda:0"):
        for name, call in _operator_calls(device):
            gpus.calls.clear()
            call()
            (called, current, args), = gpus.calls
            index = torch.device(device).index
            assert called == "matgptq_glue_" + name
            assert current == index and args[-1] == 100 + index, name
            assert gpus.current == 0  # left as it was


def test_tensors_on_different_gpus_are_refused(monkeypatch):
    gpus = _Gpus(monkeypatch)
    for name, call in _operator_calls("cuda:0", other="cuda:1"):
        with pytest.raises(_glue.GlueError, match="different GPUs"):
            call()
        assert not gpus.calls, name
