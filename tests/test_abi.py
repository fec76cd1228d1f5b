"""CPU checks of the boundary: the library loads, exports every symbol the header
declares, and the host-side mirrors validate arguments as the reference asserts."""
import os
import re

import numpy as np
import pytest

import scratchtape_amd
from scratchtape_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "scratchtape_hip.h")


def header_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(st_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_entry_points():
    syms = header_symbols()
    for name in ["st_matmul", "st_matmul_f32", "st_matmul_with", "st_ndarray_matmul", "st_softmax",
                 "st_softmax_backward", "st_knn_quantize_2bit", "st_knn_search_ivf_2bit", "st_last_error"]:
        assert name in syms


def test_library_exports_every_declared_symbol():
    L = scratchtape_amd.lib()
    for name in header_symbols():
        assert hasattr(L, name), name
    # and the Python binding covers them all with argtypes
    assert set(header_symbols()) == set(_lib.SIGNATURES)


def test_version_and_f16_switch():
    L = scratchtape_amd.lib()
    assert L.st_version().startswith(b"scratchtape_hip")
    assert L.st_f16_enabled() in (0, 1)


def test_struct_layouts_match_the_header():
    # st_matref: p, off, stride, trans, reserved, ld, group, inner
    assert _lib.StMatRef.inner.offset == 48 and _lib.ctypes.sizeof(_lib.StMatRef) == 56
    assert _lib.StEpilogue.col_sum_stride.offset == 80 and _lib.ctypes.sizeof(_lib.StEpilogue) == 88
    # st_gemm: a, b, out (st_matref), epi, batch, m, k, n, use_f16, reserved
    assert _lib.StGemm.epi.offset == 168 and _lib.StGemm.batch.offset == 256
    assert _lib.StGemm.use_f16.offset == 288 and _lib.ctypes.sizeof(_lib.StGemm) == 296


def test_null_arguments_are_rejected_without_a_device():
    L = scratchtape_amd.lib()
    rc = L.st_matmul(None, None, None, 1, 1, 1, 1, None, None)
    assert rc == _lib.ST_ERR_INVALID
    assert b"NULL" in L.st_last_error()
    rc = L.st_softmax(None, None, 4, 4, 4, 1.0, 1, 0, None)
    assert rc == _lib.ST_ERR_INVALID
    rc = L.st_matmul_grouped(None, 2, None)
    assert rc == _lib.ST_ERR_INVALID
    g = (_lib.StGemm * 2)()
    g[1].batch, g[1].m, g[1].k, g[1].n = 1, 4, 4, 4   # g[1].a.p is NULL
    rc = L.st_matmul_grouped(g, 2, None)
    assert rc == _lib.ST_ERR_INVALID and b"GEMM 0 of the group" in L.st_last_error()


def test_ndarray_matmul_shape_asserts_like_the_reference():
    from scratchtape_amd.tensor import ndarray_matmul
    with pytest.raises(ValueError, match="inner dims must match"):
        ndarray_matmul(np.zeros((2, 3), np.float32), np.zeros((4, 2), np.float32))
    with pytest.raises(ValueError, match="lhs must be 2D"):
        ndarray_matmul(np.zeros(3, np.float32), np.zeros((3, 2), np.float32))


def test_f16_route_mirrors_the_reference_pick():
    from scratchtape_amd import f16_route
    assert f16_route(128, 64, 64) and f16_route(128, 64, 96)
    assert not f16_route(70, 64, 64)          # m ragged
    assert not f16_route(64, 48, 64)          # k not a multiple of 32
    assert not f16_route(64, 64, 64, col_sum=True, b_trans=True)
    assert f16_route(4096, 256, 768)


def test_probe_arguments_are_validated_like_the_reference_asserts():
    # ivf.rs:469 asserts nprobe in 1..=min(nlist, PROBE_MAX); the width is the scan's 256.
    L = scratchtape_amd.lib()
    fake = 1 << 20  # aligned non-null stand-in: every call below is rejected before any access
    assert L.st_knn_centroid_digit_bytes(12288, 256) == 1536 * 4096
    assert L.st_knn_centroid_digit_bytes(9, 256) == 2 * 4096
    assert L.st_knn_centroid_digit_bytes(9, 128) == -1
    cases = [
        ((None, fake, fake, 64, fake, 4, 256, 8, fake, None), b"NULL"),
        ((fake, fake, fake, 64, fake, 4, 128, 8, fake, None), b"d == 256"),
        ((fake, fake, fake, 64, fake, 4, 256, 17, fake, None), b"nprobe"),
        ((fake, fake, fake, 64, fake, 4, 256, 0, fake, None), b"nprobe"),
        ((fake, fake, fake, 4, fake, 4, 256, 5, fake, None), b"nprobe"),
        ((fake, fake, fake, 64, fake + 4, 4, 256, 8, fake, None), b"aligned"),
    ]
    for args, msg in cases:
        assert L.st_knn_probe(*args) == _lib.ST_ERR_INVALID
        assert msg in L.st_last_error(), (args, L.st_last_error())
    assert L.st_knn_centroids_prep(fake, 64, 200, fake, fake, fake, None) == _lib.ST_ERR_INVALID
    assert L.st_knn_centroids_prep(fake, 0, 256, fake, fake, fake, None) == _lib.ST_ERR_INVALID


def test_fused_attention_arguments_are_validated():
    L = scratchtape_amd.lib()
    fake = 1 << 20
    for (b, h, t, hd), msg in [((32, 4, 128, 32), b"head_dim 64"), ((32, 4, 100, 64), b"multiple of 32"),
                               ((32, 4, 288, 64), b"multiple of 32"), ((0, 4, 128, 64), b"batch")]:
        assert L.st_attention_fused_fwd(fake, fake, fake, b, h, t, hd, 0.125, 0, None) == _lib.ST_ERR_INVALID
        assert msg in L.st_last_error()
        assert L.st_attention_fused_bwd(fake, fake, fake, fake, fake, b, h, t, hd, 0.125, None) == _lib.ST_ERR_INVALID
    assert L.st_attention_fused_fwd(None, fake, fake, 32, 4, 128, 64, 0.125, 0, None) == _lib.ST_ERR_INVALID


def test_layer_norm_arguments_are_validated():
    L = scratchtape_amd.lib()
    fake = 1 << 20
    assert L.st_layer_norm(None, 4, 8, fake, 0, 1e-5, 1, 0, fake, fake, fake, None) == _lib.ST_ERR_INVALID
    assert L.st_layer_norm(fake, 5, 8, fake, 0, 1e-5, 2, 16, fake, fake, fake, None) == _lib.ST_ERR_INVALID
    assert b"split evenly" in L.st_last_error()
    assert L.st_layer_norm_backward(fake, fake, fake, fake, 4, 8, fake, fake, 0, fake, 0, 2, 8, None) == \
        _lib.ST_ERR_INVALID
    assert b"overlap" in L.st_last_error()


def test_masked_search_arguments_are_validated():
    L = scratchtape_amd.lib()
    fake = 1 << 20
    assert L.st_knn_search_masked_2bit(fake, fake, 100, fake, fake, 0, 4, 256, 128, fake, fake, None) == \
        _lib.ST_ERR_INVALID
    assert b"at least 128 keys" in L.st_last_error()
    assert L.st_knn_search_masked_2bit(fake, fake, 1000, fake, fake, 0, 4, 128, 128, fake, fake, None) == \
        _lib.ST_ERR_INVALID
    assert L.st_knn_search_masked_2bit(fake, fake, 1000, fake, fake, 0, 4, 256, 129, fake, fake, None) == \
        _lib.ST_ERR_INVALID


def test_ceiling_probe_arguments_are_validated():
    L = scratchtape_amd.lib()
    fake = 1 << 20
    assert L.st_peak_mfma(5, 10, 8, fake, None) == _lib.ST_ERR_INVALID
    assert b"kind" in L.st_last_error()
    assert L.st_peak_mfma(0, 0, 8, fake, None) == _lib.ST_ERR_INVALID
    assert L.st_peak_read(fake, 24, 8, fake, None) == _lib.ST_ERR_INVALID
    assert L.st_peak_read(fake + 4, 32, 8, fake, None) == _lib.ST_ERR_INVALID
    assert L.st_lane_selftest(None, None) == _lib.ST_ERR_INVALID
    assert L.st_device_info(None, None, None, None) == _lib.ST_ERR_INVALID


def test_caller_outputs_are_size_checked_before_any_device_call():
    """A caller-supplied out smaller than what the kernel writes is refused on the host (CPU tensors: the
    check runs before the C ABI is reached)."""
    import torch

    from scratchtape_amd import rows
    from scratchtape_amd.knn import KnnStore2bit

    store = KnnStore2bit(torch.zeros((300, 64), dtype=torch.uint8), torch.ones(300), [0, 100, 300])
    q = torch.zeros((3, 256))
    probes = torch.zeros((3, 2), dtype=torch.int32)
    good = (torch.empty((3, 128), dtype=torch.int64), torch.empty((3, 128)))
    for bad in ((torch.empty((3, 127), dtype=torch.int64), good[1]), (good[0], torch.empty((2, 128))),
                (good[0], torch.empty(3 * 128))):
        with pytest.raises(ValueError, match="out"):
            store.search_ivf(q, probes, out=bad)
        with pytest.raises(ValueError, match="out"):
            store.search_masked(q, torch.zeros((3, 2), dtype=torch.int64), out=bad)
    x = torch.zeros(4 * 8)
    with pytest.raises(ValueError, match="writes 32"):
        rows.softmax(x, 4, 8, 8, 1.0, True, False, out=torch.empty(31))
    with pytest.raises(ValueError, match="writes 32"):
        rows.softmax_backward(x, x, 4, 8, 1.0, out=torch.empty(16))


def test_scratch_release_without_arenas_is_a_no_op():
    L = scratchtape_amd.lib()
    if L.st_scratch_release() != _lib.ST_OK:
        # No HIP device in this process: the call reports it instead of crashing.
        assert L.st_last_error()


def test_packed_arguments_have_the_struct_layout(monkeypatch):
    """The bytes that matmul.py packs for st_matref, st_epilogue and st_gemm, field by field, and what is refused."""
    import sys
    from scratchtape_amd import Epilogue, MatRef
    mm = sys.modules["scratchtape_amd.matmul"]
    addr = {"a": 0x7F0000000010, "b": 0x20, "o": 0x30, "bias": 0x40, "mask": 0x50, "res": 0x60}
    monkeypatch.setattr(mm, "_ptr", lambda t: addr[t])
    a = MatRef("a", 1, -2, True, 3, 4, 5)
    b, o = a.with_(h="b", trans=False), MatRef("o")
    assert (b.off, b.group, a.trans, b.trans) == (1, 4, True, False)
    epi = Epilogue(bias=("bias", 6), bias_stride=7, relu=True, mask=("mask", 8), residual=("res", 9), accumulate=True,
                   col_sum=(10, 11))
    raw = mm._pack(mm._GEMM, *a._fields(), *b._fields(), *o._fields(), *epi._fields(), 12, 13, 14, 15, 1, 0)
    assert len(raw) == _lib.ctypes.sizeof(_lib.StGemm)
    g = _lib.StGemm.from_buffer_copy(raw)
    values = lambda s: [getattr(s, f) for f, _ in s._fields_]
    assert values(g.a) == [addr["a"], 1, -2, 1, 0, 3, 4, 5] and values(g.b) == [addr["b"], 1, -2, 0, 0, 3, 4, 5]
    assert values(g.out) == [addr["o"], 0, 0, 0, 0, 0, 1, 0]
    assert values(g.epi) == [addr["bias"], 6, 7, addr["mask"], 8, addr["res"], 9, 1, 1, 1, 0, 10, 11]
    assert [g.batch, g.m, g.k, g.n, g.use_f16] == [12, 13, 14, 15, 1]
    assert mm._pack(mm._REF, *a._fields()) == raw[:56] and mm._pack(mm._EPI, *epi._fields()) == raw[168:256]
    assert mm._pack(mm._EPI, *mm._NO_EPI) == bytes(_lib.ctypes.sizeof(_lib.StEpilogue))
    assert mm._pack(mm._EPI, *Epilogue()._fields()) == bytes(_lib.ctypes.sizeof(_lib.StEpilogue))
    with pytest.raises(TypeError):
        mm._pack(mm._REF, *a.with_(off=1.5)._fields())
    with pytest.raises(TypeError):
        a.with_(offset=1)


def test_f32_attention_step_leaves_shared_buffers_to_the_separate_launches():
    """Buffers that may share memory under the separate launches' order (dS over P or dctx, ctx over the scores) are not
    taken by st_attention_fwd / _bwd, whose order differs; buffers side by side in one allocation are."""
    torch = pytest.importorskip("torch")
    from scratchtape_amd import attention
    b, h, t, hd = 1, 2, 16, 16
    n = b * h * t * t  # == b * t * h * hd
    qkv, dctx = torch.zeros(3 * n), torch.zeros(n)
    step = lambda buf, d: attention._f32_step(qkv, d, buf, b, h, t, hd, False)
    one = torch.zeros(5 * n)
    part = lambda i: one[i * n:(i + 1) * n]
    make = lambda **kw: attention.AttnBuffers(**{**dict(s=part(0), p=part(1), ctx=part(2), dp=part(3), ds=part(4),
                                                        dqkv=torch.zeros(3 * n)), **kw})
    assert step(make(), None) and step(make(), dctx)
    assert step(make(s=part(1)), None) and step(make(dp=part(4)), dctx)  # in place: each element by one thread
    assert not step(make(ctx=part(0)), None)
    assert not step(make(ds=part(1)), dctx) and not step(make(ds=one[n + n // 2:2 * n + n // 2]), dctx)
    assert not step(make(ds=dctx), dctx)


# (b h, T, head width): one-launch forms measured faster (True) or slower (False) than the separate launches.
@pytest.mark.parametrize("bh,t,hd,pays", [
    (96, 200, 80, True), (128, 128, 64, True), (384, 448, 64, True), (24, 256, 64, True), (16, 256, 64, False),
    (4, 256, 64, False), (96, 512, 64, False), (96, 500, 48, False), (96, 512, 32, True), (4, 128, 32, True),
    (8, 256, 32, False), (8, 192, 16, True), (4, 256, 16, False), (96, 448, 80, True), (96, 480, 80, False),
    (8, 256, 80, False), (64, 288, 72, False), (48, 350, 30, False), (96, 128, 96, False), (96, 448, 96, False),
    (4, 64, 128, False), (96, 384, 128, False), (96, 160, 66, False), (1, 50, 64, True)])
def test_f32_attention_takes_the_faster_launches(bh, t, hd, pays):
    from scratchtape_amd import attention
    assert attention._f32_step_pays(bh, 1, t, hd) is pays
    if bh % 4 == 0:
        assert attention._f32_step_pays(bh // 4, 4, t, hd) is pays


def test_split_work_belongs_to_the_launch_stream(monkeypatch):
    """Memory for a split search is an allocation of the stream that the launch goes to, or is not given: not for a call
    on another stream, nor for queries on another device than the current one (whose stream the launch uses)."""
    torch = pytest.importorskip("torch")
    import importlib
    import types
    knn = importlib.import_module("scratchtape_amd.knn")
    monkeypatch.setattr(knn, "_stream", lambda s: 5 if s is None else s)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch, "empty", lambda n, **kw: types.SimpleNamespace(data_ptr=lambda: 64, n=n, **kw))
    nbytes = scratchtape_amd.lib().st_knn_split_bytes(4)
    here, there = torch.device("cuda", 0), torch.device("cuda", 1)
    assert knn._split_work(4, here, None)[1:] == (64, nbytes) and knn._split_work(4, here, 5)[1:] == (64, nbytes)
    assert knn._split_work(4, here, 6) == (None, 0, 0)
    assert knn._split_work(4, there, None) == (None, 0, 0)
    assert knn._split_work(300, here, None) == (None, 0, 0)
