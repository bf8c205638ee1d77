"""nv_attention's tile form (several rows per sequence, head dim 128, blocks of
whole 16-token tiles) against the oracle, bit for bit: head groups, block
sizes, edges of tiles and of the chunks, tiles that hold rows of several
sequences, invalid rows and blocks, and values that a masked token must not let
through. Launches of few rows, the first tests' among them, take the per-row
kernels; the others bring enough rows for each size of launch."""
import time

import numpy as np
import pytest

import oracle as ora
from helpers import assert_bits_equal
from test_gpu_kernels import _attention, _attention_case, up

pytestmark = pytest.mark.gpu


def _rows(spans):
    """Flattened (positions, sequence ids) of sequences that add tokens [first, first + n)."""
    return (np.concatenate([np.arange(first, first + n) for first, n in spans]),
            np.concatenate([np.full(n, i) for i, (_, n) in enumerate(spans)]))


@pytest.mark.parametrize("qh,kvh", [(1, 1), (2, 2), (4, 2), (6, 2), (8, 2), (16, 2), (16, 1), (12, 2), (32, 1)])
@pytest.mark.parametrize("bs", [16, 48, 256])
def test_tiles_head_groups_and_block_sizes(gpu, qh, kvh, bs):
    """1, 2, 4, 8 and 16 q heads of a kv head per tile (also ratios 3, 6 and 32);
    prompts of 1, 37 and 150 tokens, so tiles hold rows of two or three sequences."""
    pos, seqs = _rows([(0, 37), (0, 1), (0, 150), (29, 5)])
    _attention_case(gpu, 300 + qh + bs, pos, seqs, qh, kvh, 128, bs, 4, -(-160 // bs), 160)


@pytest.mark.parametrize("first,n", [(0, 16), (0, 17), (15, 9), (1007, 40), (1023, 1), (1016, 8), (2040, 24), (4079, 17)])
def test_tiles_context_edges(gpu, first, n):
    """Contexts that end on, before and after the edges of 16-token tiles and of
    the 64-tile chunks, up to the longest context."""
    pos, seqs = _rows([(first, n)])
    pos, seqs = np.tile(pos, max(1, -(-4 // n))), np.tile(seqs, max(1, -(-4 // n)))
    _attention_case(gpu, 330 + n, pos, seqs, 4, 2, 128, 256, 1, 16, 4096)


@pytest.mark.parametrize("rows,first", [(600, 300), (600, 762), (300, 1000), (40, 2290)])
def test_tiles_chunk_edges_by_launch_size(gpu, rows, first):
    """With 2 kv heads of 8 q heads a launch has a block a row: more than two per CU keep 768 tokens'
    probabilities, more than one 1024, fewer 2304; contexts below and across each."""
    pos, seqs = _rows([(first, rows)])
    _attention_case(gpu, 340 + rows, pos, seqs, 16, 2, 128, 256, 1, 10, 2560)


def test_tiles_rows_in_any_order(gpu):
    """Rows of three sequences interleaved and out of order, decode rows among them."""
    rng = np.random.default_rng(350)
    pos, seqs = rng.integers(0, 500, size=67), rng.integers(0, 3, size=67)
    _attention_case(gpu, 351, pos, seqs, 4, 2, 128, 64, 3, 8, 512, q_std=6.0)


def test_tiles_invalid_rows_and_blocks(gpu):
    """Bad sequence ids and contexts give zero rows; table entries outside the
    cache drop their tokens, also in a row's last block."""
    stride, bs = 4, 64
    pos, seqs = _rows([(180, 40), (30, 40), (0, 64)])
    seqs[5], seqs[41], pos[7], pos[50] = -1, 3, 256, -1
    holes = [(1, -1), (3, 3 * stride), (stride + 1, -9), (2 * stride, 3 * stride + 4)]
    want = _attention_case(gpu, 360, pos, seqs, 4, 2, 128, bs, 3, stride, 256, holes=holes)
    assert not want[[5, 7, 41, 50]].any()


def test_tiles_masked_tokens_do_not_leak(gpu):
    """V rows of Inf, NaN and values whose products round to -0 right after a
    row's context, NaN and Inf keys, and underflowing probabilities: each row
    equals the oracle, which never reads past the context."""
    qh, kvh, dim, bs, blocks, rows = 4, 2, 128, 16, 8, 48
    q = ora.normal_bf16((rows, qh, dim), 371, 0.0, 6.0)
    kc = ora.normal_bf16((blocks, bs, kvh, dim), 372, 0.0, 1.0)
    vc = ora.normal_bf16((blocks, bs, kvh, dim), 373, 0.0, 1.0)
    flat = vc.reshape(blocks * bs, kvh, dim)  # the first row's context is tokens 0 .. 36: its sum there is -0
    flat[:37, :, 16:24], flat[0, :, 16:24], flat[37:, :, 16:24] = 0x8000, 0x8001, 0x3F80
    vc[3, 0, :, 40:48], vc[3, 5, :, 48:52], vc[3, 9, :, 52:56] = 0x7F80, 0xFF80, 0x7FC0
    kc[4, 3, 0, 7], kc[4, 5, 1, 9] = 0x7FC0, 0x7F80
    tables = np.arange(blocks, dtype=np.int32)
    pos, seqs = (np.arange(rows) + 36).astype(np.int32), np.zeros(rows, np.int32)
    want = ora.attention(q, kc, vc, pos, seqs, tables, rows, qh, kvh, dim, bs, blocks, blocks, 1, 128)
    got = _attention(gpu, q, kc, vc, pos, seqs, tables, rows, qh, kvh, dim, bs, blocks, blocks, 1, 128)
    nan = (want & 0x7FFF) > 0x7F80
    assert nan.any() and (want == 0x8000).any() and ((want & 0x7FFF) == 0x7F80).any()
    assert np.array_equal(nan, (got & 0x7FFF) > 0x7F80)  # a NaN's sign and payload are not specified
    assert_bits_equal(np.where(nan, 0, got), np.where(nan, 0, want))


@pytest.mark.parametrize("rows", [264, 1056, 2064])
def test_tiles_masked_tokens_do_not_leak_in_any_form(gpu, rows):
    """The same with launches of at most one block per CU (of 256), of at most two and of more: rows at positions 36
    .. 83 in turn, so every tile has rows that don't see all of its tokens."""
    qh, kvh, dim, bs, blocks = 4, 2, 128, 16, 8
    q = ora.normal_bf16((rows, qh, dim), 371, 0.0, 6.0)
    kc, vc = (ora.normal_bf16((blocks, bs, kvh, dim), seed) for seed in (372, 373))
    flat = vc.reshape(blocks * bs, kvh, dim)
    flat[:37, :, 16:24], flat[0, :, 16:24], flat[37:, :, 16:24] = 0x8000, 0x8001, 0x3F80
    vc[3, 0, :, 40:48], vc[3, 5, :, 48:52], vc[3, 9, :, 52:56] = 0x7F80, 0xFF80, 0x7FC0
    kc[4, 3, 0, 7], kc[4, 5, 1, 9] = 0x7FC0, 0x7F80
    tables, seqs = np.arange(blocks, dtype=np.int32), np.zeros(rows, np.int32)
    pos = (np.arange(rows) % 48 + 36).astype(np.int32)
    want = ora.attention(q, kc, vc, pos, seqs, tables, rows, qh, kvh, dim, bs, blocks, blocks, 1, 128, threads=8)
    got = _attention(gpu, q, kc, vc, pos, seqs, tables, rows, qh, kvh, dim, bs, blocks, blocks, 1, 128)
    nan = (want & 0x7FFF) > 0x7F80
    assert nan.any() and (want == 0x8000).any() and ((want & 0x7FFF) == 0x7F80).any()
    assert np.array_equal(nan, (got & 0x7FFF) > 0x7F80)
    assert_bits_equal(np.where(nan, 0, got), np.where(nan, 0, want))


@pytest.mark.parametrize("first,n", [(0, 16), (0, 17), (15, 9), (1007, 40), (1016, 8), (2040, 24), (2290, 40),
                                     (4079, 17)])
def test_tiles_context_edges_of_many_rows(gpu, first, n):
    """Edges of tiles and chunks with enough rows (80 or so, repeated) of 16 heads over 2."""
    pos, seqs = _rows([(first, n)])
    pos, seqs = np.tile(pos, -(-66 // n)), np.tile(seqs, -(-66 // n))
    _attention_case(gpu, 335 + n, pos, seqs, 16, 2, 128, 256, 1, 16, 4096)


def test_tiles_invalid_blocks_of_many_rows(gpu):
    """Table entries outside the cache at the start, in the middle and at the end of contexts."""
    stride, bs = 5, 64
    pos, seqs = _rows([(180, 120), (30, 120), (0, 160)])
    holes = [(1, -1), (3, 3 * stride), (stride + 1, -9), (2 * stride, 3 * stride + 4), (2 * stride + 2, -2)]
    _attention_case(gpu, 365, pos, seqs, 4, 2, 128, bs, 3, stride, 320, q_std=6.0, holes=holes)


MIXED = [(300, 1), (0, 70), (512, 1), (31, 1), (0, 1), (40, 2), (200, 3), (17, 15), (0, 33), (100, 1), (0, 150)]


@pytest.mark.parametrize("qh,kvh", [(1, 1), (4, 2), (8, 2), (6, 2), (16, 8), (16, 1), (32, 1)])
@pytest.mark.parametrize("bs", [16, 48, 256])
@pytest.mark.parametrize("order", ["sorted", "shuffled"])
def test_tiles_of_several_sequences(gpu, qh, kvh, bs, order):
    """One to sixteen rows a tile, one to eight sequences in it, at sequences whose first rows are first in their
    tile or not; sorted, and with every tile holding several sequences that others hold too. Some rows are invalid,
    first rows of their sequence among them, and sequence 4 has none that is valid."""
    pos, seqs = _rows(MIXED * (1 if qh > 2 else 2))
    seqs = seqs % len(MIXED)
    pos[[1, 73, 74, 75, 130]], seqs[[80, 99, 150]] = [-1, 600, -7, 4096, 5000], [-1, len(MIXED), 99]
    if order == "shuffled":
        mixed = np.random.default_rng(380).permutation(len(pos))
        pos, seqs = pos[mixed], seqs[mixed]
    _attention_case(gpu, 381 + qh + bs, pos, seqs, qh, kvh, 128, bs, len(MIXED), -(-600 // bs), 600)


def test_tiles_of_too_many_sequences_for_blocks_of_their_own(gpu):
    """600 sequences of 4 rows over 32 heads: their blocks would read more ids than a launch's bound allows, so
    tiles do all their sequences themselves."""
    pos, seqs = _rows([(i % 9, 3 + i % 3) for i in range(600)])
    assert len(pos) * 600 * 32 > 1 << 25
    _attention_case(gpu, 395, pos, seqs, 32, 32, 128, 16, 600, 1, 16)


def _attention_us(gpu, spans, qh=16, kvh=8, bs=256):
    """Best time of one launch over zeros, sequences of their own blocks, in a replayed graph of ten."""
    pos, seqs = _rows(spans)
    batch, rows, stride = len(spans), len(pos), 4096 // bs
    blocks = batch * stride
    q, cache, out = (gpu.alloc(n) for n in (rows * qh * 256, blocks * bs * kvh * 256, rows * qh * 256))
    for b in (q, cache):
        b.upload(np.zeros(b.bytes, np.uint8))
    args = (up(gpu, pos.astype(np.int32)), up(gpu, seqs.astype(np.int32)), up(gpu, np.arange(blocks, dtype=np.int32)))

    def ten():
        for _ in range(10):
            gpu.paged_attention(q, cache, cache, *args, out, rows, qh, kvh, 128, bs, blocks, stride, batch, 4096)

    ten()
    graph, best = gpu.capture(ten), float("inf")
    for _ in range(20):
        gpu.sync()
        start = time.perf_counter()
        graph.replay()
        gpu.sync()
        best = min(best, time.perf_counter() - start)
    return best * 1e5


@pytest.mark.parametrize("rows", [4, 32])
def test_tiles_leave_few_rows_to_the_decode_kernel(gpu, rows):
    """A few rows at the end of a long context take no longer as one sequence than as one sequence each. (By
    the tiles, which walk such a context alone, 154 us against 47 at 4 rows and 158 against 84 at 32.)"""
    assert _attention_us(gpu, [(4000, rows)]) < 1.3 * _attention_us(gpu, [(4000 + i, 1) for i in range(rows)])


@pytest.mark.parametrize("one,context", [(31, 4000), (7, 2000)])
def test_tiles_do_not_queue_sequences_of_one_row(gpu, one, context):
    """Sequences of one row beside a prompt cost a few times what they cost alone (2.7 and 3.8 measured): by tiles
    that walk their sequences one after the other 15 and 25 times."""
    alone = [(context, 1)] * one
    assert _attention_us(gpu, [(0, 200)] + alone) < 8 * _attention_us(gpu, alone)
