"""The decode kernel of head dim 128 (at most one block per CU, blocks of whole
64-token tiles) against the oracle, bit for bit: the edges of its 64-token V
tiles, 128-token score steps and ring of V slots, one q head and a GQA pair per
block, invalid blocks, and the slot that a fused launch writes, wherever the
row's table names it."""
import numpy as np
import pytest

import oracle as ora
from helpers import assert_bits_equal
from test_gpu_kernels import EPS, THETA, _attention_case, down, up

pytestmark = pytest.mark.gpu

EDGES = [1, 63, 64, 65, 127, 128, 129, 255, 256, 257, 320, 383, 384, 385, 448, 449, 511, 512, 513, 577, 640, 1023,
         1025, 4032, 4095, 4096]


@pytest.mark.parametrize("qh,kvh", [(2, 2), (4, 2), (6, 2), (16, 8)])
@pytest.mark.parametrize("bs", [64, 256])
def test_decode_context_edges(gpu, qh, kvh, bs):
    """One row per edge: 26 rows leave one head per block with 2 to 6 heads and a pair with 16."""
    pos = np.array(EDGES) - 1
    _attention_case(gpu, 400 + qh + bs, pos, np.arange(len(pos)), qh, kvh, 128, bs, len(pos), 4096 // bs, 4096)


@pytest.mark.parametrize("max_context", [64, 100, 640, 1000])
def test_decode_short_limits(gpu, max_context):
    """Score rows sized by the longest context allowed, also where it is no multiple of a tile."""
    pos = np.array([max_context - 1, 0, max_context // 2])
    _attention_case(gpu, 430 + max_context, pos, np.arange(3), 16, 8, 128, 64, 3, -(-max_context // 64), max_context)


@pytest.mark.parametrize("rows", [4, 20])
def test_decode_invalid_rows_and_blocks(gpu, rows):
    """Table entries outside the cache at the start, in the middle and at the end of contexts, a context with no
    valid block at all, and rows that attention skips."""
    bs, stride = 64, 16
    pos, seqs = np.full(rows, 1000), np.arange(rows)
    pos[1], seqs[2], pos[3] = 130, rows, stride * bs
    holes = [(0, -1), (7, rows * stride), (15, -3), (stride, -1), (stride + 1, -1), (stride + 2, -1)]
    want = _attention_case(gpu, 440 + rows, pos, seqs, 16, 8, 128, bs, rows, stride, 4096, holes=holes)
    assert not want[[1, 2, 3]].any()


@pytest.mark.parametrize("rows", [5, 20])
def test_decode_fused_slot_anywhere(gpu, rows):
    """The written slot is not the row's last token but an early one, in a block that the table names twice, in a
    block that it doesn't name, or invalid: out and both caches equal the oracle's, which writes first."""
    qh, kvh, dim, bs, stride, max_context = 16, 8, 128, 64, 16, 1024
    rng = np.random.default_rng(450 + rows)
    blocks = rows * (stride + 1)
    order = rng.permutation(blocks).astype(np.int32)
    tables, spare = order[:rows * stride].reshape(rows, stride).copy(), order[rows * stride:]
    pos = rng.integers(700, 1024, size=rows).astype(np.int32)
    slots = tables[:, 0] * bs + rng.integers(0, bs, size=rows).astype(np.int32)
    tables[:, 9] = tables[:, 3]
    slots[1], slots[2], slots[3] = tables[1, 3] * bs + 17, spare[2] * bs + 5, -1
    pos[4], slots[4] = 640 + 31, tables[4, 10] * bs + 31  # its own last token, as in decoding
    seqs = np.arange(rows, dtype=np.int32)
    qkv = ora.normal_bf16((rows, qh + 2 * kvh, dim), 451)
    qw, kw = ora.normal_bf16(dim, 452, 1.0, 0.02), ora.normal_bf16(dim, 453, 1.0, 0.02)
    kc0, vc0 = ora.normal_bf16((blocks, bs, kvh, dim), 454), ora.normal_bf16((blocks, bs, kvh, dim), 455)
    tb, out = gpu.alloc(max_context * dim * 4), gpu.alloc(rows * qh * dim * 2)
    gpu.rope_cache(tb, max_context, dim, THETA)
    kc, vc = up(gpu, kc0), up(gpu, vc0)
    gpu.attention_qkv_rope(*(up(gpu, a) for a in (qkv, qw, kw, pos, slots)), kc, vc, up(gpu, seqs), up(gpu, tables),
                           out, rows, qh, kvh, dim, bs, blocks, stride, rows, max_context, EPS, tb, max_context)
    q_r, k_r, v_r = ora.qkv_rope(qkv, qw, kw, pos, slots, kc0, vc0, rows, qh, kvh, dim, bs, blocks, EPS,
                                 table=down(tb, np.float32, (max_context, dim)), max_positions=max_context, threads=8)
    want = ora.attention(q_r, k_r, v_r, pos, seqs, tables, rows, qh, kvh, dim, bs, blocks, stride, rows, max_context,
                         threads=8)
    assert_bits_equal(down(kc, np.uint16, kc0.shape), k_r, "k cache")
    assert_bits_equal(down(vc, np.uint16, vc0.shape), v_r, "v cache")
    assert_bits_equal(down(out, np.uint16, (rows, qh, dim)), want, "out")
