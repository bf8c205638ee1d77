// Paged attention of decode batches at head dim 128 (attention.hip states the
// semantics and the fp32 order; this file keeps both bit for bit).
//
// A block owns one row and HPB q heads of one kv head, and has a CU to itself
// (up to 157 KB of LDS). What bounds such a launch is latency: one pass over
// the row's K, then, once the maximum is known, one serial chain of fused
// multiply-adds over its V. So the waves have roles:
//   - eight waves score, 16 tokens each per step of 128 (two per SIMD, so one
//     wave's LDS round trip hides behind the other's arithmetic), with three
//     steps of K loads in flight. They issue their first K loads as soon as the
//     row's block table is there;
//   - four waves copy V from memory straight into LDS slots of 64 tokens
//     (global_load_lds). Their queue is their own, so the first kEarlySlots tiles
//     stream in while K is still being scored;
//   - with FUSED, the first of them (the block's first wave) also does the row's q/k norm + RoPE
//     and KV-slot write, before its copies. The loads of K and V don't wait for
//     that write: the row's own slot is replaced in LDS by the values just
//     computed, wherever the block table names it.
// Then the scoring waves exponentiate, and the first 2 HPB of them run the
// value chains, one (head, dimension) a lane, the others leaving.
//   Scores: a load instruction reads whole token rows (16 lanes each); a wave
//   stages its 16 rows in LDS rows of its own, and four lanes score a token:
//   lane a of a quad owns chains 8a .. 8a + 7, so the first two tree levels
//   (offsets 16 and 8) are DPP adds over the quad, the last three in the lane.
//   Sum: thread i of 256 per head adds p_i, p_{i + 256}, ...
//   Values: tokens past the context are staged as -0.0 with p = +0, which
//   leaves every chain value unchanged; a tile of an invalid block is skipped.
//
// Measured on MI355X against four waves that take the phases in turn: 8 rows at
// contexts of 512 .. 1024 22.0 -> 19.8 us a launch (of which, for a mean of 894
// tokens, 2.5 go until q is there, 4.6 into the scores, 1.9 into maximum and
// exponentials, 5.5 into the chains and 2.5 into the launch), one row at 200
// 8.5 -> 7.0, 32 rows at 512 .. 1024 one layer in all 87.4 -> 83.5.
#include "../../include/nano_hip.h"
#include "nvr_attention.h"
#include "nvr_device.h"
#include "nvr_internal.h"

#include <type_traits>

namespace {

using nvr::kWave;
using nvr::QkvRopeArgs;

constexpr int kDim = 128;
constexpr int kScoreWaves = 8, kCopyWaves = 4;
constexpr int kThreads = (kScoreWaves + kCopyWaves) * kWave;
constexpr int kRows = 16;                    // tokens per wave and step
constexpr int kStep = kScoreWaves * kRows;   // tokens per step
constexpr int kKRow = kDim * 2 + 64;         // staged K row bytes; the pad spreads a quad's reads over the banks
constexpr int kTile = 64;                    // tokens per V tile
constexpr int kTileBytes = kTile * kDim * 2;
constexpr int kKStage = kScoreWaves * kRows * kKRow;
constexpr int kSumThreads = 256;
constexpr uint32_t kNegZeroPair = 0x80008000u;

// V slots: what 160 KB of LDS hold beside the K rows and HPB rows of 4096
// scores, and two more over the K rows once they are scored.
template <int HPB>
constexpr int kEarlySlots = HPB == 1 ? 6 : 5;
template <int HPB>
constexpr int kSlots = kEarlySlots<HPB> + kKStage / kTileBytes;

// Block barrier once this wave's LDS operations are done; vector memory
// operations (the streamed tiles, K loads in flight) stay outstanding.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Waits until at most `tiles` tiles (four loads each) of this wave are outstanding.
__device__ __forceinline__ void wait_tiles(int tiles) {
    switch (tiles) {
        case 0: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
        case 1: asm volatile("s_waitcnt vmcnt(4)" ::: "memory"); break;
        case 2: asm volatile("s_waitcnt vmcnt(8)" ::: "memory"); break;
        case 3: asm volatile("s_waitcnt vmcnt(12)" ::: "memory"); break;
        case 4: asm volatile("s_waitcnt vmcnt(16)" ::: "memory"); break;
        case 5: asm volatile("s_waitcnt vmcnt(20)" ::: "memory"); break;
        default: asm volatile("s_waitcnt vmcnt(24)" ::: "memory"); break;
    }
}

// The value chains of a row whose blocks are all valid, in inline asm: acc =
// fma(p_t, v_t[d], acc) over units of 16 tokens in order, one block barrier
// before every fourth. va is the LDS address of this lane's dimension in slot 0
// (token rows of 256 bytes, slots of 16 KB, SLOTS of them in turn), pa that of
// p_{lane % 16}.
// What bounds the chain is LDS latency over the 15 reads that lgkmcnt can tell
// apart: about 14 clocks a token (13 alone in LDS), where issue would allow 8.
// V elements are read with ds_read_u16_d16_hi into registers whose low halves
// are zero (each already is the element as an f32), the probabilities once per
// 16 tokens, lane j of each 16-lane row holding p_{16k + j}, which reach the fma
// through DPP row_newbcast:j. Reads run 12 tokens ahead (four groups of four
// registers, z), also across a tile's end: the barrier before a tile says that
// the one after it has landed too, and reads past the last tile stay inside LDS
// and are dropped. Nothing is in flight at the end. (ds_read_b64_tr_b16, four
// tokens a read but two more instructions a token to widen them, took 16 clocks
// a token.)
#define NVR_R(i, t, v) "ds_read_u16_d16_hi %[z" #i "], %[" #v "] offset:(" #t ")*256\n\t"
#define NVR_F(i, k) \
    "v_fmac_f32_dpp %[acc], %[p" #k "], %[z" #i "] row_newbcast:" #i " row_mask:0xf bank_mask:0xf\n\t"
#define NVR_RA(g, v) NVR_R(0, 4 * g, v) NVR_R(1, 4 * g + 1, v) NVR_R(2, 4 * g + 2, v) NVR_R(3, 4 * g + 3, v)
#define NVR_RB(g, v) NVR_R(4, 4 * g, v) NVR_R(5, 4 * g + 1, v) NVR_R(6, 4 * g + 2, v) NVR_R(7, 4 * g + 3, v)
#define NVR_RC(g, v) NVR_R(8, 4 * g, v) NVR_R(9, 4 * g + 1, v) NVR_R(10, 4 * g + 2, v) NVR_R(11, 4 * g + 3, v)
#define NVR_RD(g, v) NVR_R(12, 4 * g, v) NVR_R(13, 4 * g + 1, v) NVR_R(14, 4 * g + 2, v) NVR_R(15, 4 * g + 3, v)
#define NVR_P(k, o) "ds_read_b32 %[p" #k "], %[pa] offset:" #o "\n\t"
#define NVR_W(n) "s_waitcnt lgkmcnt(" #n ")\n\t"
#define NVR_FA(k) NVR_F(0, k) NVR_F(1, k) NVR_F(2, k) NVR_F(3, k)
#define NVR_FB(k) NVR_F(4, k) NVR_F(5, k) NVR_F(6, k) NVR_F(7, k)
#define NVR_FC(k) NVR_F(8, k) NVR_F(9, k) NVR_F(10, k) NVR_F(11, k)
#define NVR_FD(k) NVR_F(12, k) NVR_F(13, k) NVR_F(14, k) NVR_F(15, k)
// 16 tokens: chains groups A .. D with p_k while reading the last group of these 16 and, behind p_n at
// offset o, the first three of the next 16 (groups gd and ga, gb, gc; these from row address v).
#define NVR_16(k, gd, n, o, ga, gb, gc, v)                                                              \
    NVR_RD(gd, cur) NVR_W(12) NVR_FA(k) NVR_P(n, o) NVR_RA(ga, v) NVR_W(13) NVR_FB(k) NVR_RB(gb, v)     \
        NVR_W(13) NVR_FC(k) NVR_RC(gc, v) NVR_W(13) NVR_FD(k)
#define NVR_NEXT "s_sub_u32 %[units], %[units], 1\n\ts_cmp_eq_u32 %[units], 0\n\ts_cbranch_scc1 2f\n\t"
template <int SLOTS>
__device__ __forceinline__ float value_chain(uint32_t va, uint32_t pa, int units) {
    float acc = 0.0f, p0, p1, p2, p3;
    uint32_t z[16] = {}, cur = va, nxt = va + kTileBytes;
    int slot = 1;
    asm volatile(
        "s_waitcnt lgkmcnt(0)\n\ts_barrier\n\t"
        NVR_P(0, 0) NVR_RA(0, cur) NVR_RB(1, cur) NVR_RC(2, cur)
        "1:\n\t"
        NVR_16(0, 3, 1, 64, 4, 5, 6, cur) NVR_NEXT
        NVR_16(1, 7, 2, 128, 8, 9, 10, cur) NVR_NEXT
        NVR_16(2, 11, 3, 192, 12, 13, 14, cur) NVR_NEXT
        NVR_16(3, 15, 0, 256, 0, 1, 2, nxt) NVR_NEXT
        "v_add_u32 %[pa], 0x100, %[pa]\n\t"
        "v_mov_b32 %[cur], %[nxt]\n\t"
        "s_add_i32 %[slot], %[slot], 1\n\t"
        "s_cmp_eq_u32 %[slot], %[slots]\n\t"
        "s_cselect_b32 %[slot], 0, %[slot]\n\t"
        "v_mov_b32 %[nxt], %[slot]\n\t"
        "v_lshl_add_u32 %[nxt], %[nxt], 14, %[va]\n\t"
        "s_barrier\n\t"
        "s_branch 1b\n\t"
        "2:\n\ts_waitcnt lgkmcnt(0)\n\t"
        : [acc] "+&v"(acc), [z0] "+&v"(z[0]), [z1] "+&v"(z[1]), [z2] "+&v"(z[2]), [z3] "+&v"(z[3]),
          [z4] "+&v"(z[4]), [z5] "+&v"(z[5]), [z6] "+&v"(z[6]), [z7] "+&v"(z[7]), [z8] "+&v"(z[8]),
          [z9] "+&v"(z[9]), [z10] "+&v"(z[10]), [z11] "+&v"(z[11]), [z12] "+&v"(z[12]), [z13] "+&v"(z[13]),
          [z14] "+&v"(z[14]), [z15] "+&v"(z[15]), [p0] "=&v"(p0), [p1] "=&v"(p1), [p2] "=&v"(p2), [p3] "=&v"(p3),
          [cur] "+&v"(cur), [nxt] "+&v"(nxt), [pa] "+&v"(pa), [units] "+&s"(units), [slot] "+&s"(slot)
        : [va] "v"(va), [slots] "n"(SLOTS)
        : "memory", "scc");
    static_assert(kTileBytes == 1 << 14, "the slot's shift");
    return acc;
}
#undef NVR_R
#undef NVR_F
#undef NVR_RA
#undef NVR_RB
#undef NVR_RC
#undef NVR_RD
#undef NVR_P
#undef NVR_W
#undef NVR_FA
#undef NVR_FB
#undef NVR_FC
#undef NVR_FD
#undef NVR_16
#undef NVR_NEXT

template <int HPB, bool FUSED>
__global__ __launch_bounds__(kThreads) void attention_decode(
    const uint16_t* __restrict__ q, uint16_t* __restrict__ kc, uint16_t* __restrict__ vc,
    const int* __restrict__ positions, const int* __restrict__ seqs, const int* __restrict__ tables,
    uint16_t* __restrict__ out, int qh, int kvh, int bs, int bs_shift, int blocks, int stride, int batch,
    int max_context, int score_stride, QkvRopeArgs fa) {
    constexpr int S = kSlots<HPB>, kEarly = kEarlySlots<HPB>;
    extern __shared__ __align__(16) unsigned char smem[];
    float* probs = reinterpret_cast<float*>(smem);                  // [HPB][score_stride]
    unsigned char* vslots = smem + sizeof(float) * HPB * score_stride;  // [S][kTileBytes]
    unsigned char* kstage = vslots + kEarly * kTileBytes;               // the K rows, later the last V slots
    __shared__ __align__(16) uint16_t own[FUSED ? HPB + 2 : 1][kDim];  // this row's rotated q heads and k, and its v
    __shared__ float red_max[HPB][kScoreWaves];
    __shared__ float red_sum[HPB][kSumThreads / 32];

    // kv heads in the fastest place: blocks that lie 256 apart and share a CU one after the other are different
    // rows, and the blocks of one kv head's q heads land on one XCD (kvh a multiple of 8) and share its L2.
    const int row = blockIdx.y, kvhead = blockIdx.x, h0 = kvhead * (qh / kvh) + int(blockIdx.z) * HPB;
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int grp = lane >> 4, m16 = lane & 15;  // (FUSED, wave 0) head of the group; its lane
    const bool qgrp = grp < HPB, kgrp = grp == HPB, vgrp = grp == HPB + 1;
    uint4 xw = make_uint4(0, 0, 0, 0), nw = xw;
    if (FUSED && wave == 0) {
        __builtin_amdgcn_s_setprio(3);  // the scores wait for this wave's q
        const int hsel = qgrp ? h0 + grp : kgrp ? qh + kvhead : qh + kvh + kvhead;  // idle group: a v head
        xw = nvr::load_stream(fa.qkv + (int64_t(row) * (qh + 2 * kvh) + hsel) * kDim + 8 * m16);
        nw = *reinterpret_cast<const uint4*>((qgrp ? fa.qw : fa.kw) + 8 * m16);
    }
    const int seq = seqs[row], pos = positions[row];
    const int64_t context64 = int64_t(pos) + 1;
    const bool valid = seq >= 0 && seq < batch && context64 >= 1 && context64 <= max_context &&
                       context64 <= int64_t(stride) * bs;
    const int ctx = valid ? int(context64) : 1;
    const int64_t token_stride = int64_t(kvh) * kDim;  // elements between consecutive tokens of a block
    uint16_t* orow = out + (int64_t(row) * qh + h0) * kDim;
    int slot = -1;
    if constexpr (FUSED) {
        const int s = fa.slots[row];
        slot = s >= 0 && int64_t(s) < int64_t(bs) * blocks ? s : -1;
    }

    // Lane i of every wave holds the row's table entry i (at most 64), read back with readlane.
    int lane_entry = -1;
    if (valid && lane <= (ctx - 1) >> bs_shift) lane_entry = tables[int64_t(seq) * stride + lane];
    auto group_entry = [&](int t0) { return __builtin_amdgcn_readlane(lane_entry, min(t0, ctx - 1) >> bs_shift); };
    auto entry_ok = [&](int e) { return e >= 0 && e < blocks; };
    // First token row of an aligned group of tokens. A group past the context
    // or in an invalid block reads the first rows of block 0 instead: every
    // load stays inside an allocated block and its data is discarded.
    auto group_row = [&](int e, int t0) { return t0 < ctx && entry_ok(e) ? e * bs + (t0 & (bs - 1)) : 0; };
    const int ntiles = (ctx + kTile - 1) / kTile;

    if (wave < kCopyWaves) {
        // ---- copying waves ----
        const int cw = wave;
        const uint16_t* vcol = vc + int64_t(kvhead) * kDim;
        if constexpr (FUSED) {
            if (cw == 0) {
                // One 16-lane group per head (lane m holds elements 8m .. 8m + 7), with qkv_rope's arithmetic:
                // groups below HPB take a q head, group HPB the kv head's k, group HPB + 1 its v. With one q head
                // a block the blocks of a kv head write the same bytes. It runs for every row, as a separate
                // q/k-norm + RoPE launch would, also those that attention skips.
                const uint4 rot = nvr::qkv_rotate(fa.rope, fa.max_positions, fa.eps, xw, nw, pos, m16);
                const uint4 val = make_uint4(vgrp ? xw.x : rot.x, vgrp ? xw.y : rot.y, vgrp ? xw.z : rot.z,
                                             vgrp ? xw.w : rot.w);
                if (grp <= HPB + 1) *reinterpret_cast<uint4*>(&own[grp][8 * m16]) = val;
                if ((kgrp || vgrp) && slot >= 0)
                    nvr::store_stream((kgrp ? kc : vc) + (int64_t(slot) * kvh + kvhead) * kDim + 8 * m16, val);
                __builtin_amdgcn_s_setprio(0);
            }
        }
        if (!valid) return;
        // A tile is four 1 KB loads a wave: rows 16 cw + 4u + lane / 16, lane l landing at byte 16 l. The loads
        // are inline asm, so the compiler (which would make every later LDS read wait for all of them) never
        // sees them: wait_tiles orders them. M0 holds the LDS address and is restored after each load.
        uint32_t voff[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            voff[u] = uint32_t(((16 * cw + 4 * u + lane / 16) * int(token_stride) + 8 * (lane % 16)) * 2);
        const uint32_t slots_lds = nvr::lds_address(vslots) + cw * 4096;
        auto stream = [&](int tile, int at) {
            const uint16_t* base = vcol + int64_t(group_row(group_entry(tile * kTile), tile * kTile)) * token_stride;
            const uint32_t dst = __builtin_amdgcn_readfirstlane(slots_lds + at * kTileBytes);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                uint32_t saved;
                asm volatile(
                    "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\t"
                    "s_mov_b32 m0, %0"
                    : "=&s"(saved)
                    : "v"(voff[u]), "s"(base), "s"(dst + u * 1024)
                    : "memory");
            }
        };
        if constexpr (FUSED) lds_barrier();  // q is in LDS (before the copies: K's first loads go ahead of them)
        for (int i = 0; i < kEarly && i < ntiles; ++i) stream(i, i);
        lds_barrier();  // maxima: the K rows are free
        for (int i = kEarly; i < S && i < ntiles; ++i) stream(i, i);
        // Makes tile i whole: this wave's rows of it have landed once at most `behind` later tiles are outstanding.
        auto finish = [&](int i, int at, int behind) {
            wait_tiles(behind);
            const int t0 = i * kTile, left = ctx - t0, e = group_entry(t0);
            unsigned char* mine = vslots + at * kTileBytes + cw * 4096;
            if (FUSED && entry_ok(e)) {
                const int own_row = slot - (e * bs + (t0 & (bs - 1))) - 16 * cw;
                if (slot >= 0 && own_row >= 0 && own_row < 16 && lane < 16)
                    *reinterpret_cast<uint4*>(mine + own_row * 256 + 16 * lane) =
                        *reinterpret_cast<const uint4*>(&own[FUSED ? HPB + 1 : 0][8 * lane]);
            }
            if (left < kTile) {
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (16 * cw + 4 * u + lane / 16 >= left)
                        *reinterpret_cast<uint4*>(mine + 1024 * u + 16 * lane) =
                            make_uint4(kNegZeroPair, kNegZeroPair, kNegZeroPair, kNegZeroPair);
            }
        };
        finish(0, 0, min(ntiles, S) - 1);
        for (int i = 0, at = 0; i < ntiles; ++i) {
            const int after = at + 1 == S ? 0 : at + 1;
            // The barrier before tile i says that tile i + 1 is whole too; tiles up to i + S - 2 (S - 1 at first)
            // have been issued.
            if (i + 1 < ntiles) finish(i + 1, after, min(ntiles - 1, i == 0 ? S - 1 : i + S - 2) - (i + 1));
            lds_barrier();
            // Tile i - 1 is consumed: its slot takes the next one.
            if (i > 0 && i - 1 + S < ntiles) stream(i - 1 + S, at == 0 ? S - 1 : at - 1);
            at = after;
        }
        return;
    }

    // ---- scoring waves ----
    const int sw = wave - kCopyWaves, tid = int(threadIdx.x) - kCopyWaves * kWave;
    if (!valid) {
        for (int i = tid; i < HPB * kDim; i += kScoreWaves * kWave) orow[i] = 0;
        return;
    }
    const int tq = lane >> 2, a = lane & 3;
    const int lrow = lane / 16, lpiece = lane % 16;
    unsigned char* krows = kstage + sw * kRows * kKRow;
    const uint16_t* kcol = kc + int64_t(kvhead) * kDim + 8 * lpiece;
    const int klane = lrow * int(token_stride);
    auto first_token = [&](int s) { return s * kStep + sw * kRows; };
    // Loads are unconditional, so no branch makes the compiler drain the load queue.
    auto issue = [&](uint4 (&kb)[4], int s) {
        const int t0 = first_token(s);
        const uint16_t* base = kcol + int64_t(group_row(group_entry(t0), t0)) * token_stride;
#pragma unroll
        for (int k = 0; k < 4; ++k) kb[k] = nvr::load_stream(base + klane + 4 * k * int(token_stride));
    };
    const int nsteps = (ctx + kStep - 1) / kStep;
    uint4 kA[4], kB[4], kC[4];
    issue(kA, 0);
    issue(kB, 1);
    if constexpr (FUSED) lds_barrier();
    float qf[HPB][4][8];
#pragma unroll
    for (int g = 0; g < HPB; ++g)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            nvr::unpack8(*reinterpret_cast<const uint4*>(
                             FUSED ? &own[FUSED ? g : 0][32 * j + 8 * a]
                                   : q + (int64_t(row) * qh + h0 + g) * kDim + 32 * j + 8 * a),
                         qf[g][j]);
    const float kScale = 1.0f / sqrtf(float(kDim));
    float m[HPB];
#pragma unroll
    for (int g = 0; g < HPB; ++g) m[g] = -__builtin_inff();
    auto score = [&](const uint4 (&kb)[4], int s) {
        const int t0 = first_token(s), e = group_entry(t0);
        const bool ok = entry_ok(e);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // the previous step's reads are done
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int k = 0; k < 4; ++k) *reinterpret_cast<uint4*>(krows + (4 * k + lrow) * kKRow + 16 * lpiece) = kb[k];
        if constexpr (FUSED) {
            const int own_row = slot - (e * bs + (t0 & (bs - 1)));
            if (ok && slot >= 0 && own_row >= 0 && own_row < kRows) {  // uniform
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                if (lane < 16)
                    *reinterpret_cast<uint4*>(krows + own_row * kKRow + 16 * lane) =
                        *reinterpret_cast<const uint4*>(&own[HPB][8 * lane]);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        float kf[4][8];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            nvr::unpack8(*reinterpret_cast<const uint4*>(krows + tq * kKRow + 16 * (4 * j + a)), kf[j]);
        const int t = t0 + tq;
        const bool live = t < ctx;
#pragma unroll
        for (int g = 0; g < HPB; ++g) {
            float acc[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[i] = __builtin_fmaf(qf[g][0][i], kf[0][i], 0.0f);
#pragma unroll
            for (int j = 1; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < 8; ++i) acc[i] = __builtin_fmaf(qf[g][j][i], kf[j][i], acc[i]);
            // Offset 16: chain c + 16 = 8 (a ^ 2) + i. Offset 8: chain c + 8 = 8 (a ^ 1) + i.
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[i] += nvr::dpp<nvr::kDppQuadXor2>(acc[i]);
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[i] += nvr::dpp<nvr::kDppQuadXor1>(acc[i]);
            float dot = ((acc[0] + acc[4]) + (acc[2] + acc[6])) + ((acc[1] + acc[5]) + (acc[3] + acc[7]));
            // Pin the tree before any branch: the compiler would otherwise sink it
            // under the condition, where the DPP operands cannot be fused into their adds.
            __asm__ volatile("" : "+v"(dot));
            const float sc = live && ok ? dot * kScale : -__builtin_inff();
            m[g] = fmaxf(m[g], sc);
            if (live && a == 0) probs[g * score_stride + t] = sc;
        }
    };
    for (int s = 0; s < nsteps; s += 3) {
        issue(kC, s + 2);
        score(kA, s);
        issue(kA, s + 3);
        if (s + 1 < nsteps) score(kB, s + 1);
        issue(kB, s + 4);
        if (s + 2 < nsteps) score(kC, s + 2);
    }

    // ---- maximum, exponentials, sum ----
#pragma unroll
    for (int g = 0; g < HPB; ++g) {
        m[g] = nvr::wave_max(m[g]);
        if (lane == 0) red_max[g][sw] = m[g];
    }
    lds_barrier();
    if (sw < 4 * HPB) {  // 256 threads a head
        const int g = sw >> 2, i = tid & (kSumThreads - 1);
        float mg = red_max[g][0];
#pragma unroll
        for (int w = 1; w < kScoreWaves; ++w) mg = fmaxf(mg, red_max[g][w]);
        const bool finite = __builtin_isfinite(mg);
        float* p = probs + g * score_stride;
        float sum = 0.0f;
        // Up to four at a time: their reads and exponentials overlap.
        auto exps = [&](int t, auto count) {
            constexpr int N = decltype(count)::value;
            float pr[N];
#pragma unroll
            for (int u = 0; u < N; ++u) pr[u] = p[t + u * kSumThreads];
#pragma unroll
            for (int u = 0; u < N; ++u)
                pr[u] = finite && t + u * kSumThreads < ctx ? nvr::exp_nonpositive(pr[u] - mg) : 0.0f;
#pragma unroll
            for (int u = 0; u < N; ++u) {
                if (t + u * kSumThreads < ntiles * kTile) p[t + u * kSumThreads] = pr[u];
                sum += pr[u];  // + 0 past the context leaves it
            }
        };
        int t0 = 0;
        for (; t0 + 2 * kSumThreads < ctx; t0 += 4 * kSumThreads) exps(t0 + i, std::integral_constant<int, 4>{});
        if (t0 + kSumThreads < ctx) exps(t0 + i, std::integral_constant<int, 2>{});
        else if (t0 < ctx) exps(t0 + i, std::integral_constant<int, 1>{});
        sum = nvr::half_wave_sum(sum);
        if ((lane & 31) == 0) red_sum[g][i >> 5] = sum;
    }

    // ---- values ----
    if (sw >= 2 * HPB) {
        lds_barrier();
        return;
    }
    const int g = tid / kDim, d = tid % kDim;
    float* p = probs + g * score_stride;
    float acc = 0.0f;
    if (__ballot(lane <= (ctx - 1) >> bs_shift && !entry_ok(lane_entry)) == 0) {
        acc = value_chain<S>(nvr::lds_address(vslots) + 2 * d, nvr::lds_address(p) + 4 * (lane & 15),
                             (ctx + 15) / 16);
    } else {  // a tile of an invalid block adds no term
        for (int i = 0, at = 0; i < ntiles; ++i, at = at + 1 == S ? 0 : at + 1) {
            lds_barrier();
            if (!entry_ok(group_entry(i * kTile))) continue;
            const uint16_t* v = reinterpret_cast<const uint16_t*>(vslots + at * kTileBytes) + d;
            for (int t = 0; t < kTile; ++t) acc = __builtin_fmaf(p[i * kTile + t], nvr::bf16_to_f32(v[t * kDim]), acc);
        }
    }
    const float den = nvr::fold8(red_sum[g]);
    orow[tid] = nvr::f32_to_bf16(den > 0.0f ? acc / den : 0.0f);
}

}  // namespace

namespace nvr {

// The row's table has to fit one wave (at most 64 entries), a block to hold
// whole V tiles, and offsets inside a block to fit in int32.
bool attention_decode_fits(int bs, int kvh, int max_context) {
    return (bs & (bs - 1)) == 0 && bs >= kTile && (max_context - 1) / bs < kWave &&
           int64_t(bs) * kvh * kDim * 2 < (int64_t(1) << 31);
}

template <int HPB, bool FUSED>
void launch_attention_decode(nv_context* c, const uint16_t* q, uint16_t* k, uint16_t* v, const int* p, const int* s,
                             const int* t, uint16_t* o, int rows, int qh, int kvh, int bs, int blocks, int stride,
                             int batch, int max_context, const QkvRopeArgs& fa) {
    const int score_stride = (max_context + kTile - 1) / kTile * kTile;
    const size_t lds = sizeof(float) * HPB * score_stride + kEarlySlots<HPB> * kTileBytes + kKStage;
    hipLaunchKernelGGL((attention_decode<HPB, FUSED>), dim3(unsigned(kvh), unsigned(rows), unsigned(qh / kvh / HPB)),
                       dim3(kThreads), lds, c->stream, q, k, v, p, s, t, o, qh, kvh, bs, __builtin_ctz(unsigned(bs)), blocks, stride, batch,
                       max_context, score_stride, fa);
}

#define NVR_DECODE(HPB, FUSED)                                                                                         \
    template void launch_attention_decode<HPB, FUSED>(nv_context*, const uint16_t*, uint16_t*, uint16_t*, const int*, \
                                                      const int*, const int*, uint16_t*, int, int, int, int, int,     \
                                                      int, int, int, const QkvRopeArgs&);
NVR_DECODE(1, false)
NVR_DECODE(1, true)
NVR_DECODE(2, false)
NVR_DECODE(2, true)
#undef NVR_DECODE

}  // namespace nvr
