"""The native call path of the decode entry points against the Python one (needs an MI355X).

Both end in the same C ABI call, so wherever the native path takes a call the
results are the same bits, and what it does not take (copies of unaligned rows,
other devices and types, errors) behaves as the Python path alone does.
"""
from __future__ import annotations

import ctypes

import pytest
import torch

from engine.kernels import _native
from engine.kernels.paged_attention import paged_attention_decode_batched
from engine.kernels.paged_attention_integration import (
    paged_decode_kv_write_attention,
    paged_rope_decode_attention,
)

pytestmark = pytest.mark.gpu

B, HQ, HKV, D, BS, BLOCKS = 5, 8, 2, 64, 16, 64


def _tensors(device, form):
    """q, key, value, cos, sin in the given form, pools, tables and lengths."""
    g = torch.Generator(device=device).manual_seed(9)

    def rnd(*shape):
        return torch.randn(shape, generator=g, device=device).half()

    q, key, value = rnd(B, HQ, D), rnd(B, HKV, D), rnd(B, HKV, D)
    cos, sin = rnd(B, D), rnd(B, D)
    if form == "merged":  # slices of one projection's output
        qkv = torch.cat([q.flatten(1), key.flatten(1), value.flatten(1)], 1)
        q = qkv[:, :HQ * D].view(B, HQ, D)
        key = qkv[:, HQ * D:(HQ + HKV) * D].view(B, HKV, D)
        value = qkv[:, (HQ + HKV) * D:].view(B, HKV, D)
    elif form == "4d":  # as the attention modules hold them
        q, key, value = q.unsqueeze(2), key.unsqueeze(2), value.unsqueeze(2)
        cos, sin = cos.unsqueeze(1), sin.unsqueeze(1)
    elif form == "head_major":
        q, key, value = (t.transpose(0, 1).contiguous().transpose(0, 1) for t in (q, key, value))
    elif form == "odd":  # rows at an odd stride: copied before the launch
        q, key, value = (torch.cat([t, t[..., :1]], -1)[..., :D] for t in (q, key, value))
    pools = rnd(BLOCKS, BS, HKV, D), rnd(BLOCKS, BS, HKV, D)
    tables = torch.randperm(BLOCKS, generator=g, device=device)[:B * 12].view(B, 12).int()
    lens = torch.tensor([1, 16, 17, 100, 190], dtype=torch.int32, device=device)
    return (q, key, value, cos, sin), pools, tables, lens


def _calls(t, pools, tables, lens, name):
    q, key, value, cos, sin = t
    if name == "decode":
        return paged_attention_decode_batched(q, *pools, tables, lens, D ** -0.5)
    if name == "kv_write_decode":
        return paged_decode_kv_write_attention(q, key, value, *pools, tables, lens, D ** -0.5)
    return paged_rope_decode_attention(q, key, value, cos, sin, *pools, tables, lens, D ** -0.5)


@pytest.mark.parametrize("form", ["dense", "merged", "4d", "head_major", "odd"])
@pytest.mark.parametrize("name", ["decode", "kv_write_decode", "rope_decode"])
def test_same_bits_as_the_python_path(cuda_device, monkeypatch, name, form):
    if name == "decode" and form == "4d":
        pytest.skip("the plain call takes three dimensions")
    t, pools, tables, lens = _tensors(cuda_device, form)
    results = []
    taken = []
    native = _native.direct

    def watched(*args):
        out = native(*args)
        taken.append(out is not None)
        return out

    for direct in (lambda *a: None, watched, watched):  # the Python call sizes the workspace
        monkeypatch.setattr(_native, "direct", direct)
        own = [p.clone() for p in pools]
        out = _calls(t, own, tables, lens, name)
        results.append((out, *own))
    assert taken == [form != "odd" or name == "rope_decode"] * 2
    for got in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(got, results[0]))
        assert got[0].stride() == results[0][0].stride()


@pytest.mark.parametrize("name", ["decode", "kv_write_decode", "rope_decode"])
def test_refusals_are_the_python_checks(cuda_device, name):
    t, pools, tables, lens = _tensors(cuda_device, "dense")
    _calls(t, pools, tables, lens, name)
    for bad in (dict(tables=tables.long()), dict(lens=lens.cpu()), dict(lens=lens[:3]),
                dict(pools=(pools[0].float(), pools[1])), dict(pools=(pools[0][:9], pools[1])),
                dict(t=(t[0][:, :7], *t[1:])), dict(t=(t[0][..., :32], *t[1:]))):
        args = dict(dict(t=t, pools=pools, tables=tables, lens=lens), **bad)
        with pytest.raises(AssertionError):
            _calls(args["t"], args["pools"], args["tables"], args["lens"], name)
    with pytest.raises(AttributeError):
        _calls(t, pools, tables, lens.tolist(), name)
    empty = _calls(tuple(x[:0] for x in t), pools, tables[:0], lens[:0], name)
    assert empty.shape == (0, HQ, D)


class _Marked(torch.Tensor):
    """A subclass with __torch_function__ alone: no dispatch key tells it from a plain tensor."""


@pytest.mark.parametrize("name", ["decode", "kv_write_decode", "rope_decode"])
def test_subclasses_and_modes_take_the_python_path(cuda_device, monkeypatch, name):
    t, pools, tables, lens = _tensors(cuda_device, "dense")
    want = _calls(t, pools, tables, lens, name)
    native, taken = _native.direct, []

    def watched(*args):
        out = native(*args)
        taken.append(out is not None)
        return out

    monkeypatch.setattr(_native, "direct", watched)
    got = _calls((t[0].as_subclass(_Marked), *t[1:]), pools, tables, lens, name)
    assert type(got) is (_Marked if name == "decode" else torch.Tensor)  # empty_like keeps the type
    assert torch.equal(got.as_subclass(torch.Tensor), want)

    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert torch.equal(_calls(t, pools, tables, lens, name), want)
    assert taken == [False, False]
    parameter = torch.nn.Parameter(t[0], requires_grad=False)
    assert torch.equal(_calls((parameter, *t[1:]), pools, tables, lens, name), want)
    assert taken[-1]


# The library's status for a call it refuses before any launch, and for a HIP error.
@pytest.mark.parametrize("status", [_native.PA_ERR_ARG, _native.PA_ERR_HIP])
def test_hip_errors_are_raised_once(cuda_device, status):
    """A refused call is the Python path's to explain; a HIP error is not tried a second time."""
    t, pools, tables, lens = _tensors(cuda_device, "dense")
    want = _calls(t, pools, tables, lens, "decode")
    calls = []
    failing = ctypes.CFUNCTYPE(ctypes.c_int, *_native.SIGNATURES["pa_decode_batched_f16"][1])(
        lambda *a: calls.append(1) or status)
    module, lib = _native.host(), _native.load()
    addresses = {n: ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in module.CALLS}
    try:
        module.bind(dict(addresses, pa_decode_batched_f16=ctypes.cast(failing,
                                                                      ctypes.c_void_p).value))
        if status == _native.PA_ERR_HIP:
            with pytest.raises(_native.NativeLibraryError, match=f"status {status}"):
                _calls(t, pools, tables, lens, "decode")
        else:
            assert torch.equal(_calls(t, pools, tables, lens, "decode"), want)
    finally:
        module.bind(addresses)
    assert calls == [1]


def test_a_second_stream_gets_its_own_workspace(cuda_device):
    t, pools, tables, lens = _tensors(cuda_device, "dense")
    want = _calls(t, pools, tables, lens, "decode")
    side = torch.cuda.Stream(cuda_device)
    side.wait_stream(torch.cuda.current_stream(cuda_device))
    with torch.cuda.stream(side):
        got = [_calls(t, pools, tables, lens, "decode") for _ in range(2)]
    side.synchronize()
    assert all(torch.equal(g, want) for g in got)
    assert _native._workspaces[(cuda_device.index or 0, side.cuda_stream, _native.WS_DECODE)].is_cuda
