"""Which kernel, tile and split a GEMM call takes (st_matmul_plan), on the CPU: the dispatch that the GPU tests' shapes
rely on, seen from outside the kernels."""
import ctypes
import time

import pytest

from scratchtape_amd import _lib
from test_gemm_gpu import EDGE_F16, EDGE_F32, TILES

ANY_SHAPE, DMA, GROUP = 0, 1, 2
FORMS = [(False, False), (False, True), (True, False), (True, True)]


def plan(m, k, n, use_f16=False, ta=False, tb=False, batch=1, aligned=True, bias=False, accumulate=False,
         col_sum=False):
    """(kernel, tile rows, tile columns, slices, scratch bytes) of a call on packed matrices."""
    p = (1 << 20) + (0 if aligned else 4)
    ref = lambda trans, size: _lib.StMatRef(p, 0, size, int(trans), 0, 0, 1, 0)
    epi = _lib.StEpilogue()
    epi.bias, epi.accumulate, epi.has_col_sum = p if bias else None, int(accumulate), int(col_sum)
    out = (ctypes.c_int64 * 5)()
    _lib.check(_lib.lib().st_matmul_plan(ref(ta, m * k), ref(tb, k * n), ref(False, m * n), batch, m, k, n, epi,
                                         int(use_f16), out))
    return tuple(out)


@pytest.mark.parametrize("use_f16", [False, True])
def test_the_edge_shapes_reach_every_tile(use_f16):
    for ta, tb in FORMS:
        tiles = {}
        for shape in EDGE_F16 if use_f16 else EDGE_F32:
            kernel, *tile = plan(*shape, use_f16, ta, tb, aligned=False, bias=True)[:3]
            assert kernel == ANY_SHAPE and tuple(tile) == TILES.get(shape, tuple(tile)), (shape, ta, tb)
            tiles[tuple(tile)] = shape
        assert set(tiles) == {(32, 32), (64, 64), (128, 64) if use_f16 else (128, 128)}, (ta, tb, tiles)


# Single calls on either side of the grouped kernel's rule, at the sizes whose two times decided it (see group_of_one).
@pytest.mark.parametrize("m,k,n,use_f16,form,kernel", [
    (4096, 256, 1024, True, "nn", DMA), (4096, 256, 1024, True, "plain", DMA), (4096, 1024, 1024, True, "nt", DMA),
    (16384, 2048, 256, True, "nn", DMA), (8448, 256, 512, True, "plain", GROUP), (8448, 256, 512, True, "nn", GROUP),
    (16384, 1024, 4096, True, "nt", GROUP), (8192, 256, 1024, False, "nn", GROUP), (8192, 2048, 384, False, "nn", DMA),
    (16384, 256, 768, False, "nt", DMA), (24576, 512, 512, False, "nn", DMA), (40960, 512, 512, False, "nn", DMA),
    (57344, 512, 512, False, "nn", GROUP), (8192, 512, 2048, False, "nt", GROUP), (256, 4096, 1024, True, "tn", DMA),
    (256, 8192, 1024, True, "tn", GROUP), (1024, 1024, 4096, False, "tn", DMA), (1024, 2048, 4096, False, "tn", GROUP),
    (1024, 4096, 1024, False, "tn", GROUP), (1536, 2048, 1536, False, "tn", DMA), (1536, 4096, 1536, False, "tn", DMA),
    (768, 2048, 2304, False, "tn", GROUP), (2048, 2048, 512, True, "plain", DMA), (2048, 2048, 512, True, "tn", GROUP),
    (2048, 2048, 1024, True, "plain", GROUP)])
def test_single_calls_take_the_faster_kernel(m, k, n, use_f16, form, kernel):
    kw = dict(tn=dict(ta=True, accumulate=True, col_sum=True), nt=dict(tb=True, bias=True), nn=dict(bias=True),
              plain={})
    assert plan(m, k, n, use_f16, **kw[form])[0] == kernel


@pytest.mark.parametrize("m,k,n,ta,tb,kernel", [(1 << 20, 1024, 128, False, False, DMA),
                                                (1 << 20, 992, 128, False, True, GROUP),
                                                (1 << 20, 1024, 128, True, False, GROUP),
                                                (256, 1024, 1 << 20, False, True, DMA)])
def test_f32_operands_past_4_gib_stay_off_the_grouped_kernels_32_bit_offsets(m, k, n, ta, tb, kernel):
    assert plan(m, k, n, False, ta, tb, bias=True)[0] == kernel


def test_a_plan_needs_valid_arguments_and_no_device():
    L, out = _lib.lib(), (ctypes.c_int64 * 5)(*[9] * 5)
    ref = _lib.StMatRef(1 << 20, 0, 0, 0, 0, 0, 1, 0)
    assert L.st_matmul_plan(ref, ref, ref, 1, 8, 8, 8, None, 0, None) == _lib.ST_ERR_INVALID
    assert L.st_matmul_plan(ref, ref, None, 1, 8, 8, 8, None, 0, out) == _lib.ST_ERR_INVALID
    assert L.st_matmul_plan(ref, ref, ref, 0, 8, 8, 8, None, 0, out) == 0 and list(out) == [0] * 5


@pytest.mark.parametrize("m,k,n,slices", [(1, 1 << 20, 1, 512), (16, 1 << 20, 16, 512), (1, 1 << 24, 1, 512),
                                          (4, 100000, 4, 447), (64, 65536, 64, 128), (1, 1 << 28, 1, 512)])
def test_a_long_small_product_is_planned_in_microseconds(m, k, n, slices):
    """A small output's slice count is found without walking every possible one (k / 128 of them).  Host time of the
    whole query, ctypes included: about 4 us, which the bound leaves room for a busy machine; walking takes 60 us to
    13 ms on the shapes of 2^20 and more."""
    best = float("inf")
    for _ in range(20):
        t = time.perf_counter()
        got = plan(m, k, n, aligned=False)
        best = min(best, time.perf_counter() - t)
    assert got[:4] == (ANY_SHAPE, 32, 32, slices)
    assert best < 40e-6, best


@pytest.mark.parametrize("m,k,n", [(1, 4, 300_000_000), (31, 1, (1 << 30) - 1), (100_000, 32, 100_000),
                                   (64, 1, 1 << 27),
                                   (8_388_480, 3, 31)])
def test_large_outputs_of_small_tiles_are_accepted(m, k, n):
    """Up to 33 million 32 x 32 tiles, where the device holds the output."""
    kernel, bm, bn = plan(m, k, n, aligned=False, bias=True)[:3]
    assert (kernel, bm, bn) == (ANY_SHAPE, 32, 32) or bm > 32


def test_what_the_any_shape_kernel_refuses():
    for m, n, batch, msg in [(8_388_481, 3, 1, "8388480 rows"), (33, 5, 65536, "batch 65536"),
                             (8_388_480, (1 << 30) - 1, 1, "m = 8388480 x n = 1073741823")]:
        with pytest.raises(_lib.ScratchtapeError, match=msg):
            plan(m, 5, n, batch=batch, aligned=False, bias=True)
