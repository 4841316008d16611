"""The operators' Python side without a device: what ``torch.jit.trace``
records, and results of tensor subclasses.

The library's entry points are replaced by ones that check their arguments
against the ctypes signatures (a traced shape entry is a tensor, which they
refuse) and launch nothing.
"""

from __future__ import annotations

import pytest
import torch

import jointkv_amd as jkv
from jointkv_amd import _lib, _ops

pytestmark = pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning")


class _Recorder:
    def __init__(self):
        self.real = _lib.load()
        self.calls = []

    def __getattr__(self, name):
        if name.endswith("_workspace_bytes"):
            return getattr(self.real, name)

        def call(*args):
            types = _lib.SIGNATURES[name][1]
            assert len(types) == len(args)
            for kind, arg in zip(types, args):
                kind.from_param(arg)
            self.calls.append(name)
            return _lib.JKV_OK

        return call


@pytest.fixture
def recorder(monkeypatch):
    rec = _Recorder()
    monkeypatch.setattr(_lib, "load", lambda: rec)
    monkeypatch.setattr(_lib, "require_device", lambda *ts: next(t for t in ts if t is not None).device)
    monkeypatch.setattr(_lib, "stream_handle", lambda device: 0)
    monkeypatch.setattr(_ops, "_ROPE_CACHE", {})
    return rec


def _quantized(out):
    return out.key, out.value, out.key_indices, out.value_indices


def _exits(result):
    return (*result[0].values(), result[1])


def _calls():
    gen = torch.Generator().manual_seed(11)
    key, value = (torch.randn(1, 2, 5, 128, generator=gen).half() for _ in range(2))
    strided = torch.randn(1, 2, 128, 5, generator=gen).half().transpose(2, 3)
    query = torch.randn(1, 4, 5, 128, generator=gen).half()
    books = torch.randn(2, 16, 2, 256, 8, generator=gen)
    full = torch.randn(2, 2, 256, 128, generator=gen)
    whitener = torch.eye(128).expand(2, 128, 128).contiguous()
    eye = torch.eye(8).expand(2, 16, 8, 8).contiguous()
    gsrq = jkv.ClosedLoopUniformResidualVQ([books], [books], [None], depth=2, dynamic_bpa=2.0)
    cq = jkv.ClosedLoopGroupedCQ([books[:, :, 0]], [books[:, :, 0]], [eye], dynamic_bpa=1.0)
    cq_whitened = jkv.ClosedLoopGroupedCQ([books[:, :, 0]], [books[:, :, 0]], [eye * 2 + 0.1], dynamic_bpa=1.0)
    for codec in (gsrq, cq, cq_whitened):
        for p in codec.parameters():
            p.requires_grad_(False)
    codes = torch.zeros(1, 2, 16, 16, 2, dtype=torch.uint8)
    deployed = books.reshape(32, 2, 256, 8).half()
    lengths = torch.tensor([3], dtype=torch.int32)
    encode, pair, prefill = "jkv_rvq_encode", "jkv_rvq_encode_kv", "jkv_prefill_attention"
    # name: (call, its inputs, the entry that a replay of its trace calls again:
    # that of an autograd function; other calls are traced as their outputs)
    return {
        "grouped": (lambda x: _exits(jkv.hard_grouped_residual_vq(x, books, prefixes=(1, 2))), (key,), encode),
        "grouped, strided states and learned tables": (
            lambda x, t: _exits(jkv.hard_grouped_residual_vq(x, t, prefixes=(2,))),
            (strided, books.clone().requires_grad_()), encode),
        "full vector, fp16 tables": (lambda x, t: _exits(jkv.hard_residual_vq_exits(x, t, prefixes=(2,))),
                                     (key, full.half()), encode),
        "full vector, whitened": (
            lambda x: _exits(jkv.hard_residual_vq_exits(x, full, prefixes=(2,), assignment_whiteners=whitener)),
            (key,), encode),
        "grouped CQ": (lambda x: jkv.hard_grouped_cq(x, books[:, :, 0]), (key,), encode),
        "GSRQ codec": (lambda k, v: _quantized(gsrq(0, k, v, mode="uniform")), (key, value), pair),
        "CQ codec": (lambda k, v: _quantized(cq(0, k, v, mode="uniform")), (key, value), pair),
        "CQ codec, whitened": (lambda k, v: _quantized(cq_whitened(0, k, v, mode="uniform")), (key, value), encode),
        "prefill": (lambda q, k, v: jkv.prefill_attention(q, k, v, 0, window=64), (query, key, value), None),
        "prefill, value gradient": (lambda q, k, v: jkv.prefill_attention(q, k, v, 0, window=64),
                                    (query, key, value.clone().requires_grad_()), prefill),
        "prefill from codes": (
            lambda q: jkv.prefill_attention_from_codes(q, codes[:, :, :5], codes[:, :, :5], deployed, deployed, 0,
                                                       window=64), (query,), None),
        "prefill from codes, fused": (
            lambda q: jkv.prefill_attention_from_codes(q, codes[:, :, :5], codes[:, :, :5], deployed, deployed, 0,
                                                       window=64, fused=True), (query,), None),
        "decode": (lambda q, c: jkv.decode_attention(q, c, c, deployed, deployed, lengths, window=16, max_length=4),
                   (query[:, :, :1], codes), None),
        "decode, appending": (
            lambda q, k: jkv.decode_attention(q, codes, codes, deployed, deployed, lengths, window=16, max_length=4,
                                              key_new=k, value_new=k), (query[:, :, :1], key[:, :, :1]), None),
        "decoded window": (lambda q, w: jkv.decode_attention_window(q, w, w, lengths, window=5, max_length=4),
                           (query[:, :, :1], key), None),
        "nearest": (lambda x, t: _ops.nearest_f32(x, t),
                    (torch.randn(2, 9, 128, generator=gen), torch.randn(2, 17, 128, generator=gen)), None),
    }


@pytest.mark.parametrize("name", list(_calls()))
def test_traces(recorder, name):
    call, inputs, replayed = _calls()[name]
    eager = call(*inputs)
    traced = torch.jit.trace(call, inputs, check_trace=False)
    del recorder.calls[:]
    again = traced(*inputs)
    assert replayed is None or (recorder.calls and set(recorder.calls) == {replayed})
    eager, again = (r if isinstance(r, tuple) else (r,) for r in (eager, again))
    assert [(r.shape, r.dtype) for r in again] == [(r.shape, r.dtype) for r in eager]


class _Tagged(torch.Tensor):
    pass


@pytest.mark.parametrize("name", list(_calls()))
def test_results_are_plain_tensors(recorder, name):
    # a state's subclass is the caller's own: results do not take it on
    call, inputs, _ = _calls()[name]
    out = call(*(t.detach().as_subclass(_Tagged) for t in inputs))
    assert all(type(r) is torch.Tensor for r in (out if isinstance(out, tuple) else (out,)))
