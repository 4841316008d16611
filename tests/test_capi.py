"""C ABI checks that need no GPU: exports, signatures, argument validation."""

from __future__ import annotations

import ctypes
import re
from pathlib import Path

import pytest
import torch

from jointkv_amd import _lib

HEADER = Path(__file__).resolve().parents[1] / "include" / "jkv.h"


def _declared_functions() -> set[str]:
    text = HEADER.read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return set(re.findall(r"\b(jkv_[a-z0-9_]+)\s*\(", text))


def test_library_exports_every_declared_function():
    lib = _lib.load()
    declared = _declared_functions()
    assert "jkv_rvq_encode" in declared and "jkv_decode_attention" in declared
    for name in declared:
        assert hasattr(lib, name), f"libjkv.so does not export {name}"
    assert declared == set(_lib.SIGNATURES), "ctypes signatures out of sync with include/jkv.h"


def test_version_and_error_text():
    lib = _lib.load()
    assert lib.jkv_version() >= 100
    assert isinstance(lib.jkv_last_error(), bytes)


def _encode_call(**overrides):
    lib = _lib.load()
    args = dict(states=1, dtype=0, B=1, H=1, T=4, G=1, d=8, sb=32, sh=32, st=8, tables=1, S=1, K=256,
                whiteners=None, codes=1, cb=4, ch=4, ct=1, n_exits=0, exits=None, recon=None,
                ws=None, ws_bytes=0, stream=None)
    args.update(overrides)
    return lib.jkv_rvq_encode(*args.values())


def test_encode_rejects_invalid_geometry_before_touching_the_device():
    # These return before any HIP call, so they run without a GPU.
    assert _encode_call(K=300) == _lib.JKV_EINVAL
    assert b"256" in _lib.load().jkv_last_error()
    assert _encode_call(d=0) == _lib.JKV_EINVAL
    assert _encode_call(dtype=7) == _lib.JKV_EINVAL
    assert _encode_call(d=200) == _lib.JKV_EINVAL
    depths = (ctypes.c_int32 * 1)(5)
    assert _encode_call(n_exits=1, exits=depths, S=2) == _lib.JKV_EINVAL
    assert b"ladder" in _lib.load().jkv_last_error()
    # an empty problem is a successful no-op
    assert _encode_call(T=0) == _lib.JKV_OK


def test_workspace_queries():
    lib = _lib.load()
    assert lib.jkv_rvq_encode_workspace_bytes(8, 16, 2, 256, 8, 0) == 0
    assert lib.jkv_rvq_encode_workspace_bytes(8, 16, 2, 256, 8, 1) == 8 * 16 * 2 * 256 * 8 * 4
    # full-vector codebooks: fp16 tables + -|c|^2/2 plane + partial max norms per (head, stage)
    assert lib.jkv_rvq_encode_workspace_bytes(8, 1, 2, 256, 128, 0) == 8 * 2 * (256 * 128 * 2 + 256 * 4 + 64)
    assert lib.jkv_rvq_encode_workspace_bytes(8, 1, 33, 256, 128, 0) == 0
    assert lib.jkv_rvq_encode_workspace_bytes(8, 1, 2, 128, 128, 0) == 0
    # whitened full-vector: plus M c per codeword (fp32), M and its hi/lo planes per head
    assert lib.jkv_rvq_encode_workspace_bytes(8, 1, 2, 256, 128, 1) == (
        8 * 2 * (256 * 128 * 2 + 256 * 4 + 64) + 8 * 2 * 256 * 128 * 4 + 8 * (128 * 128 * 4 + 256 * 128 * 2))
    # whitened elsewhere: fp32 selector tables
    assert lib.jkv_rvq_encode_workspace_bytes(8, 16, 2, 256, 8, 1) == 8 * 16 * 2 * 256 * 8 * 4
    F16, BF16 = _lib.JKV_F16, _lib.JKV_BF16
    bins = 8 * 16 * 2 * 256 * 8  # [H*G,S,K,d] of the config-5 V codebooks
    # one chunk of rows: bins go straight into the gradient
    assert lib.jkv_rvq_scatter_workspace_bytes(1, 8, 512, 16, 8, 2, 256, F16, 0) == 0
    # fp16 sums are exact (fixed point), so a deterministic request needs nothing more
    assert lib.jkv_rvq_scatter_workspace_bytes(1, 8, 512, 16, 8, 2, 256, F16, 1) == 0
    # bf16 deterministic: ordered partials per 256-row chunk
    assert lib.jkv_rvq_scatter_workspace_bytes(1, 8, 512, 16, 8, 2, 256, BF16, 1) == 2 * bins * 4
    # fp16, 8-dim groups at config 5: one block per (head, group, stage)
    # already fills the chip (256 blocks), so no row chunks and no partials
    assert lib.jkv_rvq_scatter_workspace_bytes(4, 8, 2048, 16, 8, 2, 256, F16, 0) == 0
    # one stage: one block per (head, group) holds the bins, 128 blocks take
    # 2 row chunks of 4096 rows with 64-bit partials
    assert lib.jkv_rvq_scatter_workspace_bytes(4, 8, 2048, 16, 8, 1, 256, F16, 0) == bins * 8
    # bf16 (fp32 bins): one block per (head, group, stage, 8 dims) already fills the chip
    assert lib.jkv_rvq_scatter_workspace_bytes(4, 8, 2048, 16, 8, 2, 256, BF16, 0) == 0
    assert lib.jkv_rvq_scatter_workspace_bytes(4, 8, 2048, 1, 128, 2, 256, F16, 0) == 0
    # one head: 32 blocks, so 4 row chunks of 2048 rows with per-chunk partials,
    # 64-bit for fixed point and 32-bit otherwise
    head = 16 * 2 * 256 * 8
    assert lib.jkv_rvq_scatter_workspace_bytes(4, 1, 2048, 16, 8, 2, 256, F16, 0) == 4 * head * 8
    assert lib.jkv_rvq_scatter_workspace_bytes(4, 1, 2048, 16, 8, 2, 256, _lib.JKV_F32, 0) == 4 * head * 4
    # d not a multiple of 4: global atomics, no workspace
    assert lib.jkv_rvq_scatter_workspace_bytes(4, 1, 2048, 1, 6, 2, 256, F16, 0) == 0
    assert lib.jkv_decode_workspace_bytes(16, 32, 128, 4096) == 16 * 32 * 16 * 130 * 4


def test_decode_rejects_unsupported_geometry():
    # Only argument combinations that fail validation: a valid geometry with
    # placeholder pointers would launch a kernel.
    lib = _lib.load()
    rc = lib.jkv_decode_attention(1, 0, 0, 1, 1, 0, 0, 4096, 1, 1, 1, 32, 8, 8, 8, 2, 256, 1,
                                  4096, 1, 8192, 1, 1, 1 << 30, None)
    assert rc == _lib.JKV_EINVAL and b"head_dim" in lib.jkv_last_error()
    rc = lib.jkv_decode_attention(1, 0, 0, 1, 1, 0, 0, 100, 1, 1, 1, 32, 8, 16, 8, 2, 256, 1,
                                  4096, 1, 8192, 1, 1, 1 << 30, None)
    assert rc == _lib.JKV_EINVAL and b"capacity" in lib.jkv_last_error()
    rc = lib.jkv_decode_attention(1, 0, 0, 1, 1, 0, 0, 4096, 1, 1, 1, 32, 8, 16, 8, 2, 256, 1,
                                  4096, 1, 0, 1, 1, 1 << 30, None)
    assert rc == _lib.JKV_EINVAL and b"rotary" in lib.jkv_last_error()


@pytest.mark.parametrize("batch,qh,kvh,groups,stages,d,window", [
    (1, 32, 8, 16, 2, 8, 4096), (1, 32, 8, 16, 2, 8, 1501), (2, 8, 8, 16, 1, 8, 8192), (4, 32, 8, 32, 1, 4, 3000),
    (16, 32, 8, 16, 2, 8, 4096), (170, 64, 8, 16, 2, 8, 4096)])
def test_decode_takes_a_workspace_of_the_longest_splits(batch, qh, kvh, groups, stages, d, window):
    # with none the call is refused before a launch and says what it needs
    lib = _lib.load()
    rc = lib.jkv_decode_attention(16, 0, 0, 16, 16, 0, 0, window, 16, 16, batch, qh, kvh, groups, d, stages, 256, 16,
                                  window, 16, 8192, 16, 16, 0, None)
    assert rc == _lib.JKV_EINVAL
    need = int(re.search(r"needs (\d+) bytes of workspace", lib.jkv_last_error().decode()).group(1))
    assert need == batch * qh * -(-window // 2048) * 130 * 4
    assert need <= lib.jkv_decode_workspace_bytes(batch, qh, 128, window)


def test_decode_window_rejects_bad_arguments():
    # validation only: every call below fails before a launch
    lib = _lib.load()
    # capacity below the window
    rc = lib.jkv_decode_attention_window(1, 0, 0, 16, 16, 0, 0, 100, 1, 32, 8, 1, 4096, 1, 8192, 1, 1,
                                         1 << 30, None)
    assert rc == _lib.JKV_EINVAL and b"capacity" in lib.jkv_last_error()
    # rows not 16-byte aligned
    rc = lib.jkv_decode_attention_window(1, 0, 0, 18, 16, 0, 0, 4096, 1, 32, 8, 1, 4096, 1, 8192, 1, 1,
                                         1 << 30, None)
    assert rc == _lib.JKV_EINVAL and b"aligned" in lib.jkv_last_error()
    # GQA group of 3 query heads
    rc = lib.jkv_decode_attention_window(1, 0, 0, 16, 16, 0, 0, 4096, 1, 24, 8, 1, 4096, 1, 8192, 1, 1,
                                         1 << 30, None)
    assert rc == _lib.JKV_EINVAL and b"GQA" in lib.jkv_last_error()
    # workspace too small
    rc = lib.jkv_decode_attention_window(1, 0, 0, 16, 16, 0, 0, 4096, 1, 32, 8, 1, 4096, 1, 8192, 1, 1,
                                         16, None)
    assert rc == _lib.JKV_EINVAL and b"workspace" in lib.jkv_last_error()


def test_scatter_rejects_misaligned_deterministic_gradients():
    # Validation fails before any launch: the gradient pointer (2) is not
    # aligned to an 8-element fp16 slice and a deterministic sum was asked for.
    lib = _lib.load()
    grads = _lib.ptr_array(ctypes.c_void_p, [2])
    depths = _lib.ptr_array(ctypes.c_int32, [2])
    rc = lib.jkv_rvq_scatter_grad(1, grads, _lib.JKV_F16, depths, 1, 512, 256, 32, 1, 8, 8, 16,
                                  8, 2, 256, 1, 1, None, 0, None)
    assert rc == _lib.JKV_EINVAL and b"aligned" in lib.jkv_last_error()


def test_product_rejects_host_tensors_loudly():
    import jointkv_amd as jkv

    states = torch.randn(1, 2, 4, 8)
    tables = torch.randn(2, 1, 256, 8)
    with pytest.raises(ValueError, match="HIP"):
        jkv.hard_residual_vq_exits(states, tables, prefixes=(1,))


def test_nearest_rejects_rows_beyond_the_grid_before_touching_the_device():
    # one 256-thread block per 64 rows: 2^30 rows would need a 2^32-item grid
    lib = _lib.load()
    dummy = ctypes.c_void_p(16)
    for name, extra in (("jkv_nearest_f32", []), ("jkv_nearest_topk_f32", [ctypes.c_int64(2), ctypes.c_void_p(0)])):
        fn = getattr(lib, name)
        args = [dummy, ctypes.c_int64(1), ctypes.c_int64(1 << 30), ctypes.c_int64(8), dummy, ctypes.c_int64(256)]
        args += extra + [dummy, ctypes.c_void_p(0)]
        assert fn(*args) == _lib.JKV_EINVAL
        assert b"rows per head" in lib.jkv_last_error()


def test_many_job_entry_points_validate_before_touching_the_device():
    # argument errors and empty calls return before any HIP call
    lib = _lib.load()
    p = (ctypes.c_void_p * 1)(16)
    depth = (ctypes.c_int32 * 1)(1)
    bad_depth = (ctypes.c_int32 * 1)(3)
    enc = dict(n=1, states=p, dtype=0, B=1, H=1, T=4, G=1, d=8, sb=32, sh=32, st=8, tables=p, S=1, K=256,
               codes=p, cb=4, ch=4, ct=1, n_exits=1, exits=depth, recon=None, ws=None, ws_bytes=0, stream=None)

    def encode_many(**kw):
        a = dict(enc)
        a.update(kw)
        return lib.jkv_rvq_encode_many(*a.values())

    assert encode_many(n=-1) == _lib.JKV_EINVAL
    assert encode_many(K=0) == _lib.JKV_EINVAL
    assert encode_many(n_exits=99) == _lib.JKV_EINVAL
    assert encode_many(n=0) == _lib.JKV_OK
    assert encode_many(T=0) == _lib.JKV_OK
    assert encode_many(states=None) == _lib.JKV_EINVAL
    assert encode_many(exits=bad_depth) == _lib.JKV_EINVAL
    assert b"ladder" in lib.jkv_last_error()

    sc = dict(n=1, n_exits=1, grads=p, dtype=0, exits=depth, codes=p, cb=4, ch=4, ct=2, B=1, H=1, T=4, G=1,
              d=8, S=2, K=256, tables=p, accumulate=1, deterministic=0, ws=None, ws_bytes=0, stream=None)

    def scatter_many(**kw):
        a = dict(sc)
        a.update(kw)
        return lib.jkv_rvq_scatter_grad_many(*a.values())

    assert scatter_many(n=-1) == _lib.JKV_EINVAL
    assert scatter_many(K=300) == _lib.JKV_EINVAL
    assert scatter_many(dtype=7) == _lib.JKV_EINVAL
    assert scatter_many(n_exits=0) == _lib.JKV_EINVAL
    assert scatter_many(n=0) == _lib.JKV_OK
    assert scatter_many(codes=None) == _lib.JKV_EINVAL
    assert scatter_many(exits=bad_depth) == _lib.JKV_EINVAL
    # an empty problem that accumulates is a no-op
    assert scatter_many(T=0) == _lib.JKV_OK


def test_many_job_wrappers_reject_host_tensors_and_accept_empty_lists():
    from jointkv_amd import _ops

    assert _ops.rvq_encode_many([], [], groups=1, group_dim=8, exits=(1,)) == []
    assert _ops.rvq_scatter_grad_many([], (1,), [], group_dim=8) == []
    with pytest.raises(ValueError, match="HIP"):
        _ops.rvq_encode_many([torch.randn(1, 2, 4, 8).half()], [torch.randn(2, 1, 256, 8)], groups=1,
                             group_dim=8, exits=(1,))
    with pytest.raises(ValueError, match="HIP"):
        _ops.rvq_scatter_grad_many([[torch.randn(1, 2, 4, 8).half()]], (1,),
                                   [torch.zeros(1, 2, 4, 1, 1, dtype=torch.uint8)], group_dim=8,
                                   table_shape=(2, 1, 256, 8))


def _gradient_workspace_floor(name, batch, qh, kvh, tokens, window):
    """The least workspace a gradient entry takes, from its refusal of none."""
    lib = _lib.load()
    strides = (tokens * 128, tokens * 128, 128)
    rows = 4 if name == "jkv_prefill_attention_backward" else 2
    args = [x for _ in range(rows) for x in (16, *strides)]
    outs = (16, 16, 16) if rows == 4 else (16,)
    rc = getattr(lib, name)(*args, 16, *strides, 16, batch, qh, kvh, tokens, 128, 16, window, 16, 8192, *outs, 16, 0,
                            None)
    text = lib.jkv_last_error().decode()
    assert rc == _lib.JKV_EINVAL and "workspace" in text
    return int(re.findall(r"needs? (\d+)", text)[-1])


@pytest.mark.parametrize("entry,query", [
    ("jkv_prefill_attention_value_grad", "jkv_prefill_value_grad_workspace_bytes"),
    ("jkv_prefill_attention_backward", "jkv_prefill_backward_workspace_bytes")])
def test_a_gradient_workspace_serves_every_smaller_batch_and_length(entry, query):
    # shorter runs on small grids ask for more than a larger batch does; a
    # caller who sized its workspace once is served all the same
    size = getattr(_lib.load(), query)
    tokens_of = (1, 33, 192, 512, 777, 1024, 2048, 5000)
    for window in (4096, 300):
        below = [0] * len(tokens_of)
        for batch in (1, 2, 3, 8, 11, 12, 16, 40):
            floors = [_gradient_workspace_floor(entry, batch, 32, 8, t, window) for t in tokens_of]
            assert all(f <= size(batch, 32, 8, t, window) for f, t in zip(floors, tokens_of))
            assert floors == sorted(floors) and all(f >= b for f, b in zip(floors, below))
            below = floors
    # what a larger batch asks for is enough for a smaller one
    for small, large in ((1, 2), (2, 3), (11, 12), (3, 40)):
        for tokens in (192, 777, 2048):
            assert _gradient_workspace_floor(entry, small, 32, 8, tokens, 4096) <= size(large, 32, 8, tokens, 4096)


@pytest.mark.parametrize("batch,qh,kvh,tokens", [
    (1, 32, 8, 777), (1, 32, 8, 1024), (2, 32, 8, 512), (2, 32, 8, 1024), (12, 32, 8, 192), (1, 32, 4, 2048),
    (1, 32, 1, 4096), (1, 4, 4, 100)])
def test_backward_workspace_is_what_its_legs_use(batch, qh, kvh, tokens):
    lib = _lib.load()
    row = tokens * 128
    size = lib.jkv_prefill_backward_workspace_bytes(batch, qh, kvh, tokens, 4096)
    rotated = batch * (qh + kvh) * row * 2
    delta = -(-batch * qh * tokens * 4 // 256) * 256
    query_leg = batch * qh * row * 4
    value_leg = lib.jkv_prefill_value_grad_workspace_bytes(batch, qh, kvh, tokens, 4096)
    # the walk that forms both gradients: two outputs, runs of 64 rows at least
    both_legs = 2 * batch * kvh * row * 4 * -(-tokens // 64)
    area = size - delta - rotated
    assert max(query_leg, value_leg) <= area <= max(query_leg, value_leg, both_legs)
    # no factor of the key blocks' runs on the queries (it made these 2 to 5
    # times as large)
    assert size <= 150e6


@pytest.mark.parametrize("batch,qh,kvh,tokens,window", [(3, 32, 32, 364, 64), (8, 8, 8, 503, 4096), (4, 64, 32, 351, 64)])
def test_short_walks_are_not_split(batch, qh, kvh, tokens, window):
    # one query head a walk, or a window of few tiles: runs of their own would
    # cost more than they share out, so no partial slots, the rotated queries only
    size = _lib.load().jkv_prefill_value_grad_workspace_bytes(batch, qh, kvh, tokens, window)
    assert size == batch * qh * tokens * 128 * 2
