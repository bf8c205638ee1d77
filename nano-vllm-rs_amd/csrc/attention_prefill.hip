// Paged causal GQA attention over tiles of 16 (token, q head) rows on the fp32
// matrix instructions: the prefill form of nv_attention (attention.hip states
// the semantics and the fp32 order; this file keeps both bit for bit).
//
// v_mfma_f32_16x16x4_f32 computes D = C + A B as four chained fused
// multiply-adds in k order, subnormals kept (checked on MI355X over 2.5 M
// outputs, normal, widely scaled and subnormal, against host fmaf chains: no
// mismatch; the reverse order mismatches in half of them). So the two chains
// that the reference's order prescribes are matrix products:
//   - dot chain c (d = c, c + 32, c + 64, c + 96) of 16 tokens x 16 rows is one
//     instruction with k = the four d's and C = 0; the 32-lane tree over the
//     chains is 31 adds of the results;
//   - the value chain over tokens is a sequence of instructions whose k runs
//     over four consecutive tokens, accumulating in place.
// The matrix form has the FMA rate of the plain VALU on this GPU (both 34
// cycles per 1024 FMAs, and they do not overlap); what it removes is the rest:
// a row-by-row kernel reads every K and V row from LDS and widens it once per
// query row, here once per 16.
//
// Layout. A block of four waves (eight in small launches) owns 16 rows: TR = 16 >> hg_shift consecutive
// batch rows x HG = 1 << hg_shift q heads of one kv head. It does the rows of one
// sequence at a time (the others masked), so a tile of several would take them one
// after the other, whatever their contexts. Therefore a launch of several sequences
// has a block more per sequence and head group, ahead of the tiles' blocks: it does
// the tile where the sequence begins (its rows there), and the tile's block only what
// goes on from earlier tiles. Blocks find that out from the sequence ids (1 to 2 us):
// a prompt of 200 rows beside 31 sequences of one row at 4000 tokens 1236 -> 231 us (a
// block per row 211), at 300 116 -> 23; 1000 rows beside 24 at 4000 1827 -> 254; 32
// prompts of 5 rows at 300 45 -> 26; 8 prompts of 128 rows, where no tile has two, 24.3
// -> 24.9. Rows that alternate between sequences still go one after the other.
//   1. Scores, transposed (M = tokens, N = rows): wave w takes tiles of 16
//      tokens 2w, 2w + 1, 2w + 8, 2w + 9, ... Lane (m, j) holds 64 contiguous
//      bytes of token tok(m) = 4 (m % 4) + m / 4, d = 32 j .. 32 j + 31: the A
//      operands of all 32 chains. The permuted tokens make result register r
//      of lane group a the score of token 4 r + a, which is the operand layout
//      of phase 3 as it stands. The first CHUNK tiles' scores go to LDS.
//   2. Row maxima; p = exp(score - max). A wave's tiles 2w, 2w + 1 (mod 16) are
//      threads 32 w .. 32 w + 31 and 128 + 32 w .. of the reference's block
//      sum, so the sum's chains and its first five levels stay in the wave.
//   3. Values, transposed (M = d, N = rows): wave w takes d = 32 w .. 32 w + 31
//      of every tile, d = 32 w + 2 m + e in instruction e.
// Contexts longer than a chunk (64 tiles) score the later chunks a second time
// in phase 2 rather than keep them.
//
// Measured on MI355X against one block per row (attention.hip): 8 prompts of
// 1024 rows in all 80.7 -> 26.3 us, one 1021-token prompt 280 -> 64.8 us, 1024
// rows at positions 3072 .. 4095 1627 -> 517 us (58 TFLOP/s of the 140 that the
// fp32 FMAs reach; the rest is the tree, the exponentials, the second scoring of
// long contexts and, in short prompts, each block's chain of memory round trips).
//
// Masked tokens may hold anything, and must not change a row that does not see
// them. Their p is +0, so in a tile that some row sees only in part they add a
// zero of either sign: that changes nothing unless the row's value is itself a
// zero (-0 + +0), or the token holds an Inf or NaN (0 x Inf). Either way the
// tile's result is a zero or NaN in that row, and such a tile is done again on
// the VALU, token by token with the row's own mask (8 prompts of 1024 rows in
// all, where every block has such tiles: 29.3 us, 34.0 when all of them go that way).
#include "../../include/nano_hip.h"
#include "nvr_attention.h"
#include "nvr_device.h"
#include "nvr_internal.h"

namespace {

using nvr::kWave;
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kPairs = 8;    // tile pairs (mod 16 tiles) whose thread sums are the reference's warps
constexpr int kDim = 128;
constexpr int kRows = 16;    // (token, head) rows per block
constexpr int kTokens = 16;  // tokens per tile
constexpr int kMaxTiles = 4096 / kTokens;
// Sequence ids that a launch's blocks of sequences may read in all (4 bytes each, from L2: 128 MB).
constexpr int64_t kMaxScan = int64_t(1) << 25;

__device__ __forceinline__ f32x4_t mfma(float a, float b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// CHUNK = tiles whose probabilities LDS holds (1 KB each); WAVES = 4 or 8;
// SIMD_WAVES = waves per SIMD that the registers are to allow. With eight waves
// each takes one tile pair in eight and, in phase 3, one of the two
// instructions e.
template <int CHUNK, int WAVES, int SIMD_WAVES>
__global__ __launch_bounds__(WAVES * kWave, SIMD_WAVES) void attention_tiles(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
    const int* __restrict__ positions, const int* __restrict__ seqs, const int* __restrict__ tables,
    uint16_t* __restrict__ out, int rows, int qh, int kvh, int bs, int blocks, int stride, int batch, int max_context,
    int hg_shift, int row_tiles, int seq_blocks) {
    extern __shared__ __align__(16) unsigned char smem[];
    f32x4_t* probs = reinterpret_cast<f32x4_t*>(smem);  // [CHUNK][64 lanes]
    __shared__ int tile_row[kMaxTiles];                 // physical token row of each tile's first token, or -1
    __shared__ float red_max[WAVES][kRows];
    __shared__ float red_sum[kPairs][kRows];
    __shared__ uint32_t found[WAVES];
    constexpr int G = kPairs / WAVES;   // tile pairs (mod 16 tiles) per wave
    constexpr bool BOTH = WAVES == 4;   // a wave runs both instructions e
    constexpr int kThreads = WAVES * kWave;

    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int n = lane & 15, a = lane >> 4;  // row of the tile; lane group
    // Consecutive blocks take the head groups of one row tile, so each XCD
    // (blocks go round the eight) sees few kv heads and keeps their K and V in
    // its L2; the last rows, whose contexts are the longest, start first, and the
    // blocks of sequences before them (those that find nothing to do are gone at once).
    const int groups = qh >> hg_shift, per = kRows >> hg_shift;
    const int item = int(blockIdx.x) / groups, group = int(blockIdx.x) % groups;
    auto row_valid = [&](int s, int64_t ctx) {
        return s >= 0 && s < batch && ctx >= 1 && ctx <= max_context && ctx <= int64_t(stride) * bs;
    };
    const int own = item < seq_blocks ? item : -1;  // the sequence that this block is for, or -1: a tile's block
    int tile = row_tiles - 1 - (item - seq_blocks);
    if (own >= 0) {
        // The sequence's first row: kScan loads a thread in flight.
        constexpr int kScan = 4;
        uint32_t first = uint32_t(rows);
        for (int r0 = int(threadIdx.x); first == uint32_t(rows) && r0 < rows; r0 += kScan * kThreads) {
            int s[kScan];
#pragma unroll
            for (int u = 0; u < kScan; ++u) s[u] = r0 + u * kThreads < rows ? seqs[r0 + u * kThreads] : -1;
#pragma unroll
            for (int u = kScan - 1; u >= 0; --u) {
                const int r = r0 + u * kThreads;
                if (s[u] == own && row_valid(own, int64_t(positions[r]) + 1)) first = uint32_t(r);
            }
        }
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) first = min(first, nvr::xor_lane_bits(first, o));
        if (lane == 0) found[wave] = first;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < WAVES; ++w) first = min(first, found[w]);
        if (first == uint32_t(rows)) return;
        tile = __builtin_amdgcn_readfirstlane(int(first)) / per;
    }
    const int head = (group << hg_shift) + (n & ((1 << hg_shift) - 1));
    const int kvhead = (group << hg_shift) / (qh / kvh);
    const int row = tile * per + (n >> hg_shift);
    const bool exists = row < rows;
    const int seq_n = exists ? seqs[row] : -1;
    const int64_t ctx64 = exists ? int64_t(positions[row]) + 1 : 0;
    const bool valid = exists && row_valid(seq_n, ctx64);
    uint32_t todo = uint32_t(__ballot(valid)) & 0xffffu;  // rows still to do (the same in every wave)
    if (own >= 0) {
        todo &= uint32_t(__ballot(seq_n == own));
    } else if (seq_blocks != 0 && todo != 0) {
        // The tile's first sequence mostly goes on from the row before; of the others, this block does those that an
        // earlier tile has seen.
        const int lead = __builtin_amdgcn_readlane(seq_n, __builtin_ctz(todo));
        const int before = tile * per - 1;
        const bool goes_on = before >= 0 && seqs[before] == lead && row_valid(lead, int64_t(positions[before]) + 1);
        const uint32_t rest = goes_on ? todo & ~uint32_t(__ballot(seq_n == lead)) : todo;
        if (rest != 0) {
            uint32_t seen = 0;
            for (int r = int(threadIdx.x); r < tile * per; r += kThreads) {
                const int s = seqs[r];
                uint32_t same = 0;
#pragma unroll
                for (int i = 0; i < kRows; ++i) same |= uint32_t(s == __builtin_amdgcn_readlane(seq_n, i)) << i;
                if ((same & rest) != 0 && row_valid(s, int64_t(positions[r]) + 1)) seen |= same;
            }
#pragma unroll
            for (int o = 1; o < kWave; o <<= 1) seen |= nvr::xor_lane_bits(seen, o);
            if (lane == 0) found[wave] = seen;
            __syncthreads();
#pragma unroll
            for (int w = 0; w < WAVES; ++w) seen |= found[w];
            todo &= ~rest | uint32_t(__builtin_amdgcn_readfirstlane(int(seen)));
        }
    }
    const int64_t row_head = int64_t(exists ? row : 0) * qh + head;
    const int wd = BOTH ? wave : wave >> 1, e = BOTH ? 0 : wave & 1;  // dimensions 32 wd ..; (one) instruction
    uint16_t* dst = out + row_head * kDim + 32 * wd + 8 * a;
    if (own < 0 && exists && !valid) *reinterpret_cast<uint4*>(dst) = make_uint4(0, 0, 0, 0);

    float qf[32];  // q[32 a + c]: operand B of chain c
#pragma unroll
    for (int i = 0; i < 4; ++i)
        nvr::unpack8(*reinterpret_cast<const uint4*>(q + row_head * kDim + 32 * a + 8 * i), qf + 8 * i);
    const float kScale = 1.0f / sqrtf(float(kDim));
    const int64_t token_stride = int64_t(kvh) * kDim;
    const uint16_t* kcol = kc + int64_t(kvhead) * kDim;
    const uint16_t* vcol = vc + int64_t(kvhead) * kDim;
    const int klane = (4 * (n & 3) + (n >> 2)) * int(token_stride) + 32 * a;

    while (todo != 0) {
        const int seq = __builtin_amdgcn_readlane(seq_n, __builtin_ctz(todo));
        const bool active = valid && seq_n == seq;
        todo &= ~uint32_t(__ballot(active));
        const int ctx = active ? int(ctx64) : 0;
        int hi = ctx, lo = active ? ctx : max_context;
#pragma unroll
        for (int o = 1; o < kRows; o <<= 1) {
            hi = max(hi, nvr::xor_lane(hi, o));
            lo = min(lo, nvr::xor_lane(lo, o));
        }
        const int ctx_max = __builtin_amdgcn_readfirstlane(hi), ctx_min = __builtin_amdgcn_readfirstlane(lo);
        const int tiles = (ctx_max + kTokens - 1) / kTokens, full = ctx_min / kTokens;
        if (int(threadIdx.x) < tiles) {
            const int t0 = int(threadIdx.x) * kTokens, lb = t0 / bs;
            const int entry = tables[int64_t(seq) * stride + lb];
            tile_row[threadIdx.x] = entry >= 0 && entry < blocks ? entry * bs + (t0 - lb * bs) : -1;
        }
        __syncthreads();

        // Tiles past the context or in an invalid block load the first rows
        // of block 0; their scores are masked and their values skipped.
        auto place = [&](int t) { return __builtin_amdgcn_readfirstlane(tile_row[min(t, tiles - 1)]); };
        auto load_k = [&](uint4 (&kb)[4], int t) {
            const uint16_t* base = kcol + int64_t(max(place(t), 0)) * token_stride;
#pragma unroll
            for (int i = 0; i < 4; ++i) kb[i] = *reinterpret_cast<const uint4*>(base + klane + 8 * i);
        };
        auto scores = [&](const uint4 (&kb)[4], int t) -> f32x4_t {
            const uint32_t* w = reinterpret_cast<const uint32_t*>(kb);
            auto chain = [&](int c) {
                return mfma(c & 1 ? nvr::bf16_hi(w[c >> 1]) : nvr::bf16_lo(w[c >> 1]), qf[c], f32x4_t{0, 0, 0, 0});
            };
            auto l16 = [&](int c) { return chain(c) + chain(c + 16); };
            auto l8 = [&](int c) { return l16(c) + l16(c + 8); };
            auto l4 = [&](int c) { return l8(c) + l8(c + 4); };
            auto l2 = [&](int c) { return l4(c) + l4(c + 2); };
            const f32x4_t dot = l2(0) + l2(1);
            const bool ok = place(t) >= 0;
            f32x4_t s;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                s[r] = ok && t * kTokens + 4 * r + a < ctx ? dot[r] * kScale : -__builtin_inff();
            return s;
        };
        // Wave-tile s of this wave: the pair 2w, 2w + 1 of every 2 WAVES tiles.
        auto tile_of = [&](int s) { return 2 * WAVES * (s >> 1) + 2 * wave + (s & 1); };

        // ---- 1. scores and row maxima ----
        float m = -__builtin_inff();
        {
            uint4 kA[4], kB[4];
            load_k(kA, tile_of(0));
            load_k(kB, tile_of(1));
            auto step = [&](uint4 (&kb)[4], int s) {
                const int t = tile_of(s);
                const f32x4_t sc = scores(kb, t);
                load_k(kb, tile_of(s + 2));
#pragma unroll
                for (int r = 0; r < 4; ++r) m = fmaxf(m, sc[r]);
                if (t < CHUNK) probs[t * kWave + lane] = sc;
            };
            for (int s = 0; tile_of(s) < tiles; s += 2) {
                step(kA, s);
                if (tile_of(s + 1) < tiles) step(kB, s + 1);
            }
        }
        m = fmaxf(m, nvr::xor_lane(m, 16));
        m = fmaxf(m, nvr::xor_lane(m, 32));
        if (a == 0) red_max[wave][n] = m;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < WAVES; ++w) m = fmaxf(m, red_max[w][n]);
        const bool finite = __builtin_isfinite(m);

        float sums[G][2][4] = {};           // the reference's thread sums of this wave's tiles (mod 16)
        f32x4_t o0 = {0, 0, 0, 0}, o1 = {0, 0, 0, 0};
        for (int c0 = 0; c0 < tiles; c0 += CHUNK) {
            const int c1 = min(tiles, c0 + CHUNK);
            // ---- 2. probabilities of the chunk ----
            auto prob = [&](f32x4_t sc, int t, float (&sum)[4]) {
                f32x4_t p;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    p[r] = finite ? nvr::exp_nonpositive(sc[r] - m) : 0.0f;
                    sum[r] += p[r];
                }
                probs[(t - c0) * kWave + lane] = p;
            };
            if (c0 == 0) {
                for (int s = 0; tile_of(s) < c1; s += 2 * G) {
#pragma unroll
                    for (int u = 0; u < 2 * G; ++u) {
                        const int t = tile_of(s + u);
                        if (t < c1) prob(probs[t * kWave + lane], t, sums[u >> 1][u & 1]);
                    }
                }
            } else {
                const int s0 = c0 / WAVES;
                uint4 kA[4], kB[4];
                load_k(kA, tile_of(s0));
                load_k(kB, tile_of(s0 + 1));
                for (int s = s0; tile_of(s) < c1; s += 2 * G) {
#pragma unroll
                    for (int u = 0; u < 2 * G; ++u) {
                        const int t = tile_of(s + u);
                        uint4(&kb)[4] = u & 1 ? kB : kA;
                        if (t < c1) {
                            const f32x4_t sc = scores(kb, t);
                            load_k(kb, tile_of(s + u + 2));
                            prob(sc, t, sums[u >> 1][u & 1]);
                        }
                    }
                }
            }
            __syncthreads();

            // ---- 3. values of the chunk ----
            auto load_v = [&](uint32_t (&v)[4], int t) {
                const uint16_t* base = vcol + int64_t(max(place(t), 0)) * token_stride + 32 * wd + 2 * n;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    v[r] = *reinterpret_cast<const uint32_t*>(base + (4 * r + a) * int(token_stride));
            };
            // Token by token, each row masked by its own context.
            auto masked = [&](int t) {
                const uint16_t* base = vcol + int64_t(place(t)) * token_stride + 32 * wd + 8 * a;
                const float* pt = reinterpret_cast<const float*>(probs + (t - c0) * kWave);
                const int end = min(kTokens, ctx_max - t * kTokens);
#pragma unroll 1
                for (int i = 0; i < end; ++i) {
                    const float p = pt[(16 * (i & 3) + n) * 4 + (i >> 2)];
                    const bool sees = t * kTokens + i < ctx;
                    float f[8];
                    nvr::unpack8(*reinterpret_cast<const uint4*>(base + i * int(token_stride)), f);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float x = __builtin_fmaf(p, e ? f[2 * r + 1] : f[2 * r], o0[r]);
                        o0[r] = sees ? x : o0[r];
                        if constexpr (BOTH) {
                            const float y = __builtin_fmaf(p, f[2 * r + 1], o1[r]);
                            o1[r] = sees ? y : o1[r];
                        }
                    }
                }
            };
            auto chains = [&](const uint32_t (&v)[4], int t, f32x4_t& x, f32x4_t& y) {
                const f32x4_t p = probs[(t - c0) * kWave + lane];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    x = mfma(nvr::bf16_hi(v[r] << (e ? 0 : 16)), p[r], x);
                    if constexpr (BOTH) y = mfma(nvr::bf16_hi(v[r]), p[r], y);
                }
            };
            auto values = [&](const uint32_t (&v)[4], int t) {
                if (place(t) >= 0) chains(v, t, o0, o1);  // an invalid block adds no term
            };
            const int f1 = min(full, c1);
            uint32_t vA[4], vB[4], vC[4], vD[4];
            load_v(vA, c0);
            load_v(vB, c0 + 1);
            load_v(vC, c0 + 2);
            int t = c0;
            for (; t + 3 < f1; t += 4) {
                load_v(vD, t + 3);
                values(vA, t);
                load_v(vA, t + 4);
                values(vB, t + 1);
                load_v(vB, t + 5);
                values(vC, t + 2);
                load_v(vC, t + 6);
                values(vD, t + 3);
            }
            // The last few, and the tiles that some row sees only in part.
            for (; t < c1; ++t) {
                load_v(vD, t + 3);
                if (place(t) >= 0) {
                    f32x4_t x = o0, y = o1;
                    chains(vA, t, x, y);
                    bool lost = false;
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        lost |= !(__builtin_fabsf(x[r]) > 0.0f) || (BOTH && !(__builtin_fabsf(y[r]) > 0.0f));
                    if (t >= full && __ballot(lost && active) != 0) {
                        masked(t);
                    } else {
                        o0 = x;
                        o1 = y;
                    }
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    vA[r] = vB[r];
                    vB[r] = vC[r];
                    vC[r] = vD[r];
                }
            }
            if (c1 < tiles) __syncthreads();  // the next chunk overwrites the probabilities
        }

        // ---- 4. the block sum's tree and the output ----
        // Tile pair (2w, 2w + 1): offset 16 between the two tiles, 8 and 4
        // between registers r, 2 and 1 between lane groups a.
#pragma unroll
        for (int g = 0; g < G; ++g) {
            float x[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) x[r] = sums[g][0][r] + sums[g][1][r];
            float s = (x[0] + x[2]) + (x[1] + x[3]);
            s += nvr::xor_lane(s, 32);
            s += nvr::xor_lane(s, 16);
            if (a == 0) red_sum[WAVES * g + wave][n] = s;
        }
        __syncthreads();
        const float den = ((red_sum[0][n] + red_sum[4][n]) + (red_sum[2][n] + red_sum[6][n])) +
                          ((red_sum[1][n] + red_sum[5][n]) + (red_sum[3][n] + red_sum[7][n]));
        if constexpr (BOTH) {
            float o[8];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                o[2 * r] = den > 0.0f ? o0[r] / den : 0.0f;
                o[2 * r + 1] = den > 0.0f ? o1[r] / den : 0.0f;
            }
            if (active) *reinterpret_cast<uint4*>(dst) = nvr::pack8(o);
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (active) dst[2 * r + e] = nvr::f32_to_bf16(den > 0.0f ? o0[r] / den : 0.0f);
        }
        if (todo != 0) __syncthreads();  // the next sequence reuses the LDS arrays
    }
}

}  // namespace

namespace nvr {

// Rows of one sequence share a tile's K and V; a batch of one row per sequence
// would leave 15 of 16 rows masked and walk its sequences one after the other,
// so the batch must average at least four rows a sequence (64 sequences of 4 rows
// at 1000 tokens 175 -> 77 us, 4 of 4 23 -> 73 by the tiles).
//
// A tile walks its context alone, in the time of one row or of sixteen, so few
// rows are better off spread over the CUs. At blocks that attention_decode takes
// (16 q heads over 8; one row a block, then tiles, us): 8 rows at 64 tokens 5.3,
// 9.8, at 1024 15, 39, at 4000 46, 153; 32 rows 6.1, 9.9, then 18, 39 and 56, 154.
// Up to two blocks per CU, by attention_ordered, one sequence still gains at short
// contexts (64 rows: 8.2, 9.9, then 40, 39 and 143, 154); several, whose K and V are
// as many times the bytes, gain less there (4 prompts of 20 rows 8.4, 9.7) than they
// lose at others (at 300 tokens 24, 19; 8 of 8 rows at 1024 56, 40). Other block sizes take attention_ordered,
// which is slower: 16-token blocks, 16 rows 9.5, 9.9, at 2000 70, 68, 32 rows 10.2, 9.9
// and 79, 69.
bool attention_tiles_fit(const nv_context* c, int rows, int qh, int kvh, int dim, int bs, int batch,
                         int max_context) {
    if (dim != kDim || bs % kTokens != 0 || rows < 4 * int64_t(batch)) return false;
    const int64_t cus = c->cu_count > 0 ? c->cu_count : 256, heads = int64_t(rows) * qh;
    if (!attention_decode_fits(bs, kvh, max_context)) return heads > cus;
    const int64_t row_blocks = (qh / kvh) % 2 == 0 ? heads / 2 : heads;
    return row_blocks > (batch == 1 ? 2 * cus : cus);
}

void launch_attention_tiles(nv_context* c, const uint16_t* q, const uint16_t* k, const uint16_t* v, const int* p,
                            const int* s, const int* t, uint16_t* o, int rows, int qh, int kvh, int bs, int blocks,
                            int stride, int batch, int max_context) {
    const int ratio = qh / kvh;
    int shift = 0;
    while (shift < 4 && ratio % (2 << shift) == 0) ++shift;
    const int per = kRows >> shift, row_tiles = (rows + per - 1) / per, groups = qh >> shift;
    const int seq_blocks = batch > 1 && int64_t(batch) * rows * groups <= kMaxScan ? batch : 0;
    const unsigned grid = unsigned(row_tiles + seq_blocks) * unsigned(groups);
    auto launch = [&](auto kernel, int chunk, int waves) {
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(unsigned(waves * kWave)),
                           sizeof(f32x4_t) * chunk * kWave, c->stream, q, k, v, p, s, t, o, rows, qh, kvh, bs, blocks,
                           stride, batch, max_context, shift, row_tiles, seq_blocks);
    };
    // Three blocks a CU hide more of each other's latency than two, and score more
    // of a long context twice (48 tiles are 768 tokens): with three per CU to fill
    // them 1021 tokens take 68.6 against 73.0 us, 2 x 512 44.1 against 50.3, 1024 at
    // 3072 518 against 525 (8 x 128 29.3 against 28.4). A launch of at most one
    // block per CU keeps 2304 tokens' scores instead, and has eight waves a block:
    // 64 tokens at 2000 103 -> 91.7 -> 69.7 us, one prompt of 256 16.5 -> 14.9. The
    // sequences' blocks count there, where a second round would cost as much as the
    // first (8 prompts of 30 rows 9.4 us, by eight waves 15.1), but not above (some do
    // nothing; 64 sequences of 8 rows at 1000 tokens 128 us, by three blocks a CU 139).
    const unsigned tiles = unsigned(row_tiles) * unsigned(groups);
    const unsigned cus = c->cu_count > 0 ? unsigned(c->cu_count) : 256u;
    if (tiles > 2 * cus) launch(attention_tiles<48, 4, 3>, 48, 4);
    else if (grid > cus) launch(attention_tiles<64, 4, 2>, 64, 4);
    else launch(attention_tiles<144, 8, 2>, 144, 8);
}

}  // namespace nvr
