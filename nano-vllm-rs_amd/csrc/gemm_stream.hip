// GEMM of few rows over a wide weight: Y[m, n] = bf16(X[m, k] W[n, k]^T), fp32
// accumulation, m <= 32 (nv_gemm's decode shapes: the tied head, qkv, gate_up).
//
// Such a product is the stream of W. What decides its rate is how W is read: in
// the matrix instructions' operand layout a load takes 64 bytes of each of 16
// rows, and half lines stream at 5.2 TB/s here, whole ones at up to 6.6. So W
// goes through LDS: global_load_lds brings four rows x 256 bytes an
// instruction, straight from memory, and the operands are read from there.
//
// Layout. A block per CU of eight waves walks tiles of 16 columns (rows of W).
// Wave w owns the k range [w k/8, (w + 1) k/8): its X operands stay in registers
// for all tiles, and its part of a tile, in units of 16 rows x 128 k (4 KB),
// passes through kRing LDS slots of its own, so no barrier is needed before the
// matrix instructions (A = W, B = X: lane l holds four consecutive columns of
// row l % 16). Slots keep a row's sixteen 16-byte pieces in the order p ^ row, which the
// copy's addresses produce, so a wave's reads of one piece of 16 rows fall into
// different banks. The eight partial tiles are summed in wave order through
// two LDS buffers in turn (one barrier a tile), by waves in turn while the
// others go on. The order is fixed, so every launch of a shape gives the same
// bits.
//
// Measured on MI355X against hipBLAS (us a launch in graphs over three weights of
// normal values, W cold): n 151936, k 1024 at 8 rows 62.2 -> 53.4 and at 32 rows
// 75.6 -> 59.8 (5.2 TB/s of W); kernel time in a decode step of 8 rows 57.7 -> 50.3;
// n 4096, k 1024 at 32 rows 8.4 -> 4.7; n 6144 8.5 -> 6.0. Four slots a wave instead of three change
// nothing; operands read from memory in their own layout take 58.9 us at one row
// of n 151936 (here 52) and 118 at 32.
#include "nvr_device.h"
#include "nvr_internal.h"

namespace {

using nvr::kWave;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8, kThreads = kWaves * kWave;
constexpr int kTileN = 16;
constexpr int kUnitK = 128;                  // k of a unit
constexpr int kUnitBytes = kTileN * kUnitK * 2;
constexpr int kRing = 3;                     // units in flight per wave (96 KB per CU)

// At most `units` units (four loads each) of this wave outstanding.
__device__ __forceinline__ void wait_units(int units) {
    static_assert(kRing <= 4, "the counts below");
    switch (units) {
        case 0: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
        case 1: asm volatile("s_waitcnt vmcnt(4)" ::: "memory"); break;
        case 2: asm volatile("s_waitcnt vmcnt(8)" ::: "memory"); break;
        default: asm volatile("s_waitcnt vmcnt(12)" ::: "memory"); break;
    }
}

// MT = row tiles of X (16 rows each); KS = k / 1024.
template <int MT, int KS>
__global__ __launch_bounds__(kThreads) void gemm_stream(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                        uint16_t* __restrict__ y, int m, int n) {
    constexpr int K = kWaves * kUnitK * KS, STEPS = kUnitK / 32;
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int i = lane & 15, j = lane >> 4;  // operand row; k group
    unsigned char* ring = smem + wave * (kRing * kUnitBytes);
    f32x4_t* red = reinterpret_cast<f32x4_t*>(smem + kWaves * kRing * kUnitBytes);  // [2][kWaves][MT][64]

    const int tiles = n / kTileN;
    // This block's tiles lie side by side (>= 1), so the 32-byte pieces of Y's rows fill lines in one XCD's L2.
    const int first = int(int64_t(blockIdx.x) * tiles / gridDim.x);
    const int mine = int(int64_t(blockIdx.x + 1) * tiles / gridDim.x) - first;
    const int units = mine * KS;
    // Copy u of a unit: rows 4u + lane / 16, the piece that belongs to slot lane % 16.
    uint32_t off[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int r = 4 * u + j;
        off[u] = uint32_t(r * K * 2 + (i ^ r) * 16);
    }
    const uint32_t ring_lds = __builtin_amdgcn_readfirstlane(nvr::lds_address(ring));
    const uint16_t* wk = w + wave * (kUnitK * KS);
    // The loads are inline asm, so the compiler (which would make every later LDS read wait for all of them) never
    // sees them: wait_units orders them. M0 holds the LDS address and is restored after each load.
    auto copy = [&](int unit, int at) {
        const uint16_t* base = wk + int64_t(first + unit / KS) * (kTileN * K) + (unit % KS) * kUnitK;
        const uint32_t dst = ring_lds + at * kUnitBytes;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            uint32_t saved;
            asm volatile(
                "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt\n\t"
                "s_mov_b32 m0, %0"
                : "=&s"(saved)
                : "v"(off[u]), "s"(base), "s"(dst + u * 1024)
                : "memory");
        }
    };
    bf16x8_t xv[MT][KS][STEPS];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int row = min(t * 16 + i, m - 1);  // rows past m repeat the last one and are not written
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int s = 0; s < STEPS; ++s)
                xv[t][ks][s] = *reinterpret_cast<const bf16x8_t*>(x + int64_t(row) * K + (wave * KS + ks) * kUnitK +
                                                                  32 * s + 8 * j);
    }
    for (int u = 0; u < kRing && u < units; ++u) copy(u, u);

    int at = 0;
    for (int q = 0; q < mine; ++q) {
        f32x4_t acc[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int unit = q * KS + ks;
            wait_units(min(units - 1 - unit, kRing - 1));
            const unsigned char* row = ring + at * kUnitBytes + i * 256;
            bf16x8_t wv[STEPS];
#pragma unroll
            for (int s = 0; s < STEPS; ++s) wv[s] = *reinterpret_cast<const bf16x8_t*>(row + ((4 * s + j) ^ i) * 16);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot is read
            if (unit + kRing < units) copy(unit + kRing, at);
            at = at + 1 == kRing ? 0 : at + 1;
#pragma unroll
            for (int s = 0; s < STEPS; ++s)
#pragma unroll
                for (int t = 0; t < MT; ++t)
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[s], xv[t][ks][s], acc[t], 0, 0, 0);
        }
        f32x4_t* part = red + (q & 1) * (kWaves * MT * kWave);
#pragma unroll
        for (int t = 0; t < MT; ++t) part[(wave * MT + t) * kWave + lane] = acc[t];
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // leaves the copies in flight
        const int t = (wave - q * MT) & (kWaves - 1);  // the waves take turns
        if (t < MT) {
            f32x4_t sum = part[t * kWave + lane];
#pragma unroll
            for (int v = 1; v < kWaves; ++v) sum += part[(v * MT + t) * kWave + lane];
            const int row = t * 16 + i;
            const int n0 = (first + q) * kTileN + 4 * j;
            if (row < m)
                *reinterpret_cast<uint2*>(y + int64_t(row) * n + n0) =
                    make_uint2(nvr::pack_bf16x2(sum[0], sum[1]), nvr::pack_bf16x2(sum[2], sum[3]));
        }
    }
}

template <int MT, int KS>
void launch(nv_context* c, const uint16_t* x, const uint16_t* w, uint16_t* y, int m, int n, int cus) {
    const size_t lds = kWaves * kRing * kUnitBytes + sizeof(f32x4_t) * 2 * kWaves * MT * kWave;
    hipLaunchKernelGGL((gemm_stream<MT, KS>), dim3(unsigned(cus)), dim3(kThreads), lds, c->stream, x, w,
                       y, m, n);
}

}  // namespace

namespace nvr {

// From as many tiles as CUs every CU has a stream; with fewer, gemm_narrow and
// gemm_rows (gemm.hip) or the library split the work further.
bool gemm_stream_fits(const nv_context* c, const void* x, const void* w, const void* y, int m, int n, int k) {
    const int cus = c->cu_count > 0 ? c->cu_count : 256;
    return m >= 1 && m <= 32 && n > 0 && n % kTileN == 0 && n / kTileN >= cus && (k == 1024 || k == 2048) &&
           aligned(x, 16) && aligned(w, 16) && aligned(y, 8);
}

void launch_gemm_stream(nv_context* c, const uint16_t* x, const uint16_t* w, uint16_t* y, int m, int n, int k) {
    const int cus = c->cu_count > 0 ? c->cu_count : 256;
    if (k == 1024) m <= 16 ? launch<1, 1>(c, x, w, y, m, n, cus) : launch<2, 1>(c, x, w, y, m, n, cus);
    else m <= 16 ? launch<1, 2>(c, x, w, y, m, n, cus) : launch<2, 2>(c, x, w, y, m, n, cus);
}

}  // namespace nvr
