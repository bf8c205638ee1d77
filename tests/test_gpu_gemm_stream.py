"""The few-row GEMMs: over a wide weight (nv_gemm and nv_gemm_rows from as many
16-column tiles as CUs) against the float64 product: one and two row tiles with
ragged last ones, both k, one tile a block and ragged numbers of tiles, more
units than the ring's slots, and equal bits from launch to launch."""
import time

import numpy as np
import pytest

import oracle as ora
from helpers import assert_bits_equal
from test_gpu_kernels import _gemm_bound, down, f32_of, up

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 15, 16, 17, 32])
@pytest.mark.parametrize("k", [1024, 2048])
@pytest.mark.parametrize("extra", [0, 1, 255, 700])
def test_gemm_stream_within_bound(gpu, m, k, extra):
    n = 16 * (gpu.sm_count() + extra)
    xa = ora.normal_bf16((m, k), m + k + extra)
    wa = ora.normal_bf16((n, k), m + k + extra + 1, 0.0, 0.05)
    x, w, y = up(gpu, xa), up(gpu, wa), up(gpu, np.full((m + 1, n), 0x7FC0, np.uint16))
    gpu.gemm(x, w, y, m, n, k)
    got = down(y, np.uint16, (m + 1, n)).copy()
    assert (got[m] == 0x7FC0).all()  # nothing past the last row
    want, bound = _gemm_bound(xa, wa)
    assert np.all(np.abs(f32_of(got[:m]).astype(np.float64) - want) <= bound)
    for call in (gpu.gemm, gpu.gemm_rows):
        call(x, w, y, m, n, k)
        assert_bits_equal(down(y, np.uint16, (m + 1, n))[:m], got[:m])


@pytest.mark.parametrize("m", [1, 8, 16, 17, 31, 32])
@pytest.mark.parametrize("n,k", [(16, 1024), (1024, 2048), (1008, 3072), (2032, 1024), (48, 4096)])
def test_gemm_narrow_within_bound(gpu, m, n, k):
    """Fewer 16-column tiles than CUs: 8-column tiles from 17 rows, through both entry points."""
    xa = ora.normal_bf16((m, k), m + n + k)
    wa = ora.normal_bf16((n, k), m + n + k + 1, 0.0, 0.05)
    x, w = up(gpu, xa), up(gpu, wa)
    want, bound = _gemm_bound(xa, wa)
    for call in (gpu.gemm, gpu.gemm_rows):
        y = up(gpu, np.full((m + 1, n), 0x7FC0, np.uint16))
        call(x, w, y, m, n, k)
        got = down(y, np.uint16, (m + 1, n))
        assert (got[m] == 0x7FC0).all()
        assert np.all(np.abs(f32_of(got[:m]).astype(np.float64) - want) <= bound)


@pytest.mark.parametrize("m,n,k", [(8, 8192, 1024), (8, 1024, 2048), (32, 1024, 2048), (64, 1024, 1024)])
@pytest.mark.parametrize("null", [0, 1, 2])
def test_gemm_refuses_a_null_operand(gpu, m, n, k, null):
    """On the host, whichever kernel the shape takes."""
    buffers = [gpu.alloc(2 * size) for size in (m * k, n * k, m * n)]
    args = [None if i == null else b.ptr for i, b in enumerate(buffers)]
    assert gpu.lib.nv_gemm(gpu._device.ctx, *args, m, n, k) == -2
    assert b"required" in gpu.lib.nv_last_error()
    gpu.sync()


def _gemm_us(gpu, call, m, n, k):
    """Best time of one product over zeros, in a replayed graph of twenty."""
    x, w, y = (gpu.alloc(2 * size) for size in (m * k, n * k, m * n))
    for b in (x, w):
        b.upload(np.zeros(b.bytes, np.uint8))

    def twenty():
        for _ in range(20):
            call(x, w, y, m, n, k)

    twenty()
    graph, best = gpu.capture(twenty), float("inf")
    for _ in range(20):
        gpu.sync()
        start = time.perf_counter()
        graph.replay()
        gpu.sync()
        best = min(best, time.perf_counter() - start)
    return best * 5e4


@pytest.mark.parametrize("k", [2048, 4096])
def test_gemm_rows_take_one_round_of_blocks(gpu, k):
    """One 16-column tile more than fit as 8-column tiles, a block per CU, costs little more than the last that fit
    (in 8-column tiles, two rounds of blocks, half as much again)."""
    n = 8 * gpu.sm_count()
    assert _gemm_us(gpu, gpu.gemm_rows, 32, n + 16, k) < 1.3 * _gemm_us(gpu, gpu.gemm_rows, 32, n, k)


@pytest.mark.parametrize("m,n,k", [(16, 4080, 3072), (16, 3584, 4096), (24, 512, 2048), (32, 256, 2048)])
def test_gemm_leaves_to_the_library_what_it_does_faster(gpu, m, n, k):
    """Few rows, but more bytes of X in all the blocks than of W, or products that the library splits over k."""
    assert _gemm_us(gpu, gpu.gemm, m, n, k) < 0.92 * _gemm_us(gpu, gpu.gemm_rows, m, n, k)


@pytest.mark.parametrize("m,n,k", [(16, 3072, 2048), (16, 3088, 2048), (9, 1920, 3072), (16, 1936, 3072),
                                   (16, 2048, 4096), (16, 2064, 4096), (8, 4080, 4096), (17, 1136, 1024),
                                   (32, 1152, 1024), (17, 560, 2048), (32, 576, 2048)])
def test_gemm_around_the_library_s_sizes(gpu, m, n, k):
    """The last product on either side of each line of the rule."""
    xa = ora.normal_bf16((m, k), m + n + k)
    wa = ora.normal_bf16((n, k), m + n + k + 1, 0.0, 0.05)
    y = up(gpu, np.full((m + 1, n), 0x7FC0, np.uint16))
    gpu.gemm(up(gpu, xa), up(gpu, wa), y, m, n, k)
    got = down(y, np.uint16, (m + 1, n))
    assert (got[m] == 0x7FC0).all()
    want, bound = _gemm_bound(xa, wa)
    assert np.all(np.abs(f32_of(got[:m]).astype(np.float64) - want) <= bound)


@pytest.mark.parametrize("m", [17, 32])
@pytest.mark.parametrize("k", [1024, 2048, 3072, 4096])
def test_gemm_rows_around_one_round_of_blocks(gpu, m, k):
    """The last n of 8-column tiles and the first of 16-column ones."""
    for n in (8 * gpu.sm_count(), 8 * gpu.sm_count() + 16):
        xa = ora.normal_bf16((m, k), m + n + k)
        wa = ora.normal_bf16((n, k), m + n + k + 1, 0.0, 0.05)
        y = up(gpu, np.full((m + 1, n), 0x7FC0, np.uint16))
        gpu.gemm_rows(up(gpu, xa), up(gpu, wa), y, m, n, k)
        got = down(y, np.uint16, (m + 1, n))
        assert (got[m] == 0x7FC0).all()
        want, bound = _gemm_bound(xa, wa)
        assert np.all(np.abs(f32_of(got[:m]).astype(np.float64) - want) <= bound)
