// Skinny-M (M <= 64) fused dequant-GEMM forward: the HBM-bound decode/rollout regime.
//
//   y[M, N] = x[M, K] . deq(W)^T + bias + s * (x . A^T) . B^T          (W FLAT [N, K])
//
// Every byte of the packed weight is read from HBM exactly once, decoded in registers to the exact bf16 value of the
// reference decoder and fed to v_mfma_f32_16x16x32_bf16 against x fragments.  Two launches for up to four forwards on one x
// (q + k + v, gate + up), no atomics, no zeroed buffers, fixed summation orders (deterministic):
//
//  1. stream_split_kernel: a grid of (row block) x (K split) tiles, one block of 8 waves per compute unit (two where the tile is
//     small).  The block owns 16 RT weight rows, each wave an eighth of the split's K range of all of them: a wave brings its x and its
//     weights into a part of LDS that is its own, by direct-to-LDS loads of whole 128-byte row pieces that run ahead, and waits for
//     them by count, so nothing in the stream waits for another wave.  The eight waves' sums meet in LDS at the end.  What a block
//     moves beside its weights is x (2 M K_b bytes, from the L2) and one fp32 partial sum per output and split.  One wave each of
//     some blocks forms the low-rank parts x . A^T on the way.
//  2. stream_epilogue_kernel: sums the splits in order, adds bias and s * su . B^T in fp32 and rounds once to bf16; for gate
//     and up of an MLP it writes h = SwiGLU(gate, up) of the two rounded outputs instead.
//
// The split of K depends on a forward's own shape only: a joint launch gives the bits of the separate ones.
//
// What bounds it: at 64 rows and RT 6 about 5 us until the first weights are there (half of a wave's rows at once in the order in which
// they are multiplied), 14 for products that the vector units' decode bounds (19 instructions and four MFMAs per 8 weights a lane,
// two waves a SIMD), 4 until the slowest wave is done and the sums have met: gate | up of 4096 -> 2 x 12288 takes 27 us in int4
// (50 MB), 31 in block-fp8 (100 MB), 35 in nf4 (two rounds of three row tiles), and the epilogue 9.5; at few rows the fixed costs of two
// dependent launches.  Before, waves owned rows, K was split between five to sixteen blocks, and fragments were loaded straight to
// registers: 32 + 13 and 36 + 13 us.  Forward of one projection at r 16, weights from memory, us, against that (24 / 48 / 64 rows):
//     int4 [12288, 4096] 17.1 22.2 23.3 -> 16.5 17.8 20.6    [4096, 4096] 14.1 14.6 15.9 -> 11.0 12.4 13.5    [2944, 7808] 17.4 -> 16.6 at 64
//     fp8  [12288, 4096] 18.6 21.1 21.9 -> 17.6 19.2 22.2    [4096, 4096] 15.0 15.2 16.4 -> 12.6 15.1 14.8    [1024, 4096] 12.7 -> 11.2 at 64
//     nvfp4 [12288, 4096], 64 rows 24.0 -> 21.8, nf4 27.3 -> 22.3; of the MLP 4096 / 12288 of 64 rows: int4 64.9 -> 57.2, fp8 69.0 -> 64.4
#include <stdlib.h>

#include <algorithm>
#include <atomic>

#include "xq_common.h"
#include "xq_lora.h"
#include "xq_skinny.h"

namespace xq {

constexpr int kStreamJobs = 4;
constexpr int kStreamWaves = 8;          // of a block

struct StreamJob {
    const uint8_t* packed;
    const uint8_t* scales;
    const float* global_scale;
    const void* lora_A;        // [r, K] fp32 or bf16
    float* partial;            // [splits][M][N]
    float* su_part;            // [K / 128][M][r_pad]
    int32_t N, group, scale_dtype;
    int32_t splits;            // K splits
    int32_t chunk_q, chunk_rem; // 128-element steps per split: chunk_q, one more in the first chunk_rem splits
    int32_t row_blocks;
    int32_t lora_f32, r, r_pad;
};
struct StreamBatch {
    StreamJob job[kStreamJobs];
};

// how a lane gets the scales of its codes: four steps' bf16 scales of int4 groups of 128 in one load, four steps' 8 scale bytes (nvfp4
// e4m3, nf4 fp32) dealt over the row's four lanes, one per half step or per fragment, requested a half step ahead, or (block-fp8) one
// value per row tile and step from registers
enum { kScFp8 = 0, kScInt4Window = 1, kScDealt = 2, kScHalf = 3, kScUse = 4 };

// scales lie where their elements may: a pair of words from any byte (one global_load_dwordx2 like an aligned one)
typedef u32x2 u32x2_a1 __attribute__((aligned(1)));

// bytes of LDS beside the waves' parts: the levels of nf4
constexpr int stream_levels(int fmt) { return fmt == XQ_FMT_NF4 ? 64 : 0; }
// Whether half a step of x (16 MT rows) and 128 bytes of 16 RT weight rows for each wave fit a block's LDS, and whether two such blocks share
// a compute unit (more tiles are too many registers for that).
constexpr bool stream_fits(int levels, int mt, int rt) { return kStreamWaves * 2048 * (mt + rt) + levels <= 160 * 1024; }
constexpr bool stream_pairs(int levels, int mt, int rt) { return mt < 4 && mt * rt <= 4 && kStreamWaves * 2048 * (mt + rt) + levels <= 80 * 1024; }

// What a wave keeps in LDS: XB half steps of x (16 MT rows of 64 elements each) and WB units of weights (128 bytes of each of its 16 RT
// rows: a step of block-fp8, two steps of the 4-bit formats).
template <int FMT, int MT, int RT>
struct StreamGeo {
    static constexpr int HPW = FMT == XQ_FMT_FP8 ? 2 : 4;          // half steps of a weight unit
    static constexpr int XH = MT * 2048, WU = RT * 2048;
    static constexpr bool PAIR = stream_pairs(stream_levels(FMT), MT, RT);
    static constexpr int ROOM = ((PAIR ? 80 : 160) * 1024 - stream_levels(FMT)) / kStreamWaves;
    static constexpr int XB = 3 * XH + 2 * WU <= ROOM ? 3 : 2 * XH + WU <= ROOM ? 2 : 1;
    static constexpr int WB = XB * XH + 2 * WU <= ROOM ? 2 : 1;
    static constexpr int WAVE = XB * XH + WB * WU;
    static constexpr int NX = 2 * MT, NW = 2 * RT;                 // loads of a half step of x, of a weight unit
    static constexpr int EARLY = RT > 1 ? RT / 2 : 1;              // row tiles that the first half step waits for at its start
    static_assert(WAVE <= ROOM, "the wave's LDS");
    // Half step v requests x of v + XB and, once the unit's last step has gone to registers, the weight unit WB ahead
    static constexpr bool issues_w(int v) { return (v & (HPW - 1)) == HPW - 2; }
    // loads requested ahead beside the first half step's own
    static constexpr int spare() {
        int n = 0;
        for (int v = -(XB > WB * HPW ? XB : WB * HPW); v < 0; ++v) n += (v + XB > 0 ? NX : 0) + (issues_w(v) && (v + 2) / HPW - 1 + WB > 0 ? NW : 0);
        return n;
    }
    // Loads that may still be out when half step h starts: those requested after the last of what it reads.
    static constexpr int ahead(int h) {
        int x = issues_w(h - XB) ? NW : 0;
        for (int v = h - XB + 1; v < h; ++v) x += NX + (issues_w(v) ? NW : 0);
        return h & (HPW - 1) || x < behind_w() ? x : behind_w();
    }
    // loads requested between a weight unit and its first half step
    static constexpr int behind_w() {
        int w = 0;
        for (int v = HPW - 1 - WB * HPW; v < 0; ++v) w += NX + (issues_w(v) ? NW : 0);
        return w;
    }
};

template <int FMT, int SC, int MT, int RT>
__global__ void __launch_bounds__(64 * kStreamWaves, (StreamGeo<FMT, MT, RT>::PAIR ? 4 : 2))
stream_split_kernel(const bf16_t* x, int64_t ldx, int32_t M, int32_t K, int32_t first1, int32_t first2, int32_t first3, StreamBatch b) {
    using G = StreamGeo<FMT, MT, RT>;
    constexpr int EB = FMT == XQ_FMT_FP8 ? 1 : 2;                 // elements per byte
    constexpr int HPW = G::HPW, XB = G::XB, WB = G::WB;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, lr = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int bx = blockIdx.x;
    const int ji = (bx >= first1 ? 1 : 0) + (bx >= first2 ? 1 : 0) + (bx >= first3 ? 1 : 0);
    const StreamJob& g = b.job[ji];
    const int at = bx - (ji == 0 ? 0 : ji == 1 ? first1 : ji == 2 ? first2 : first3);
    const int split = at % g.splits, rb = at / g.splits;
    // this wave's steps: an eighth of the split's
    const int s_begin = split * g.chunk_q + (split < g.chunk_rem ? split : g.chunk_rem);
    const int s_steps = g.chunk_q + (split < g.chunk_rem ? 1 : 0);
    const int per = s_steps / kStreamWaves, rem = s_steps % kStreamWaves;
    const int c_begin = s_begin + wave * per + (wave < rem ? wave : rem);
    const int n_steps = per + (wave < rem ? 1 : 0);
    const int k_begin = c_begin << 7;

    // ---- the low-rank parts x . A^T: units of (step, 16 ranks), dealt over the split's blocks so that a block has one for one of its
    // waves at most unless the weight is narrow.  A's operand of a wave's first unit is requested with the first loads and waits in
    // registers as bf16; the product is made of the x fragments that the stream reads anyway and goes out step by step (ranks >= r:
    // whatever row 0 gives, never read).
    const int rank_tiles = g.r_pad >> 4;
    int su_unit = rb, su_step = 1 << 30, su_tile = 0;
    const auto next_unit = [&]() {                                 // this wave's next one of units rb, rb + row_blocks, ...
        const int before = c_begin - s_begin;
        su_step = 1 << 30;
        for (; rank_tiles && su_unit < (before + n_steps) * rank_tiles; su_unit += g.row_blocks) {
            const int step = su_unit / rank_tiles - before;
            if (step >= 0) {
                su_step = step;
                su_tile = su_unit - (step + before) * rank_tiles;
                su_unit += g.row_blocks;
                break;
            }
        }
    };
    u32x4 a[4];
    const auto load_a = [&]() {
        const int row = su_tile * 16 + lr;
        const int64_t base = (int64_t)(row < g.r ? row : 0) * K + k_begin + su_step * 128 + q * 16;
        if (g.lora_f32) {
            const float* p = (const float*)g.lora_A + base;
            f32x4 raw[8];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                raw[2 * j] = *(const f32x4*)(p + (j >> 1) * 64 + (j & 1) * 8);
                raw[2 * j + 1] = *(const f32x4*)(p + (j >> 1) * 64 + (j & 1) * 8 + 4);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
                a[j] = u32x4{pack_bf16x2(raw[2 * j][0], raw[2 * j][1]), pack_bf16x2(raw[2 * j][2], raw[2 * j][3]),
                             pack_bf16x2(raw[2 * j + 1][0], raw[2 * j + 1][1]), pack_bf16x2(raw[2 * j + 1][2], raw[2 * j + 1][3])};
        } else {
            const bf16_t* p = (const bf16_t*)g.lora_A + base;
#pragma unroll
            for (int j = 0; j < 4; ++j) a[j] = *(const u32x4*)(p + (j >> 1) * 64 + (j & 1) * 8);
        }
    };

    // ---- this wave's LDS and what comes into it.  x: half step of [16 MT rows][8 pieces of 8 elements], piece p of row m at p ^ ((m >> 1)
    // & 5); weights: [16 RT rows][8 pieces of 16 bytes], piece p of row n at p ^ (n >> 1 & 7).  Lane l of a load lands at piece l of its
    // KB, so the swizzle is applied to the address that it fetches; eight neighbouring lanes take 128 bytes of a row, which a load in
    // the fragments' order does not: that one takes 56 clocks of the address unit, this one 16.  (Weights 64 bytes at a time, as
    // 16 rows of a load, read 100 MB in 24.8 us where this takes 18.4.)
    const int row0 = rb * (16 * RT) < g.N ? rb * (16 * RT) : g.N - 16;   // tiles of 16 (N % 16 == 0: a tile is all in or all out; one past the end repeats the last)
    const uint32_t xl = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem + wave * G::WAVE, wl = xl + XB * G::XH;
    const unsigned char* xs = smem + wave * G::WAVE;
    const unsigned char* wsm = xs + XB * G::XH;
    // rows of x in groups of eight: (rows past M repeat the last one: their products are never stored)
    const int tail = (M - 1) & ~7, xr = lane >> 3;
    const uint32_t x_full = (uint32_t)((int64_t)xr * ldx * 2), x_tail = (uint32_t)((int64_t)(tail + xr < M ? xr : M - 1 - tail) * ldx * 2);
    const uint32_t xc0 = ((lane & 7) ^ ((lane >> 4) & 1)) << 4, xc1 = xc0 ^ 64;
    const int halves = 2 * n_steps;
    const auto issue_x1 = [&](int h_, int x_slot, int i) {
        const int h = h_ < halves ? h_ : halves - 1;
        const bool whole = i * 8 + 8 <= M;
        const bf16_t* base = x + (int64_t)(whole ? i * 8 : tail) * ldx + k_begin + h * 64;
        const uint32_t off = (whole ? x_full : x_tail) + (i & 1 ? xc1 : xc0);
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     :: "s"(__builtin_amdgcn_readfirstlane(xl + x_slot * G::XH + i * 1024)), "v"(off), "s"(base) : "memory");
    };
    uint32_t w_off[RT];
    {
        const int n = lane >> 3, piece = (lane & 7) ^ (lane >> 4);    // rows n and n + 8 of a tile: the swizzle's bit 2 is the row's bit 3
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) w_off[rt] = (uint32_t)((int64_t)((row0 + rt * 16 < g.N ? rt * 16 : g.N - 16 - row0) + n) * (K / EB) + piece * 16);
    }
    const uint32_t w_flip = ((lane & 7) ^ (lane >> 4)) & 4 ? (uint32_t)-64 : 64u, w_rows8 = (uint32_t)(8 * (K / EB)) + w_flip;
    const uint8_t* w_base = g.packed + ((int64_t)row0 * K + k_begin) / EB;
    const int w_bytes = n_steps * (128 / EB), units = (w_bytes + 127) >> 7;
    const auto issue_w1 = [&](int u_, int slot, int i) {
        const int u = u_ < units ? u_ : units - 1;
        const uint8_t* base = w_base + (int64_t)u * 128;
        uint32_t off = w_off[i >> 1] + (i & 1 ? w_rows8 : 0);
        // (an odd step at the end of a 4-bit range: the unit's second half is fetched from the first)
        if (EB == 2 && u * 128 + 128 > w_bytes) off -= ((lane & 7) ^ (lane >> 4) ^ (i & 1 ? 4 : 0)) & 4 ? 64 : 0;
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     :: "s"(__builtin_amdgcn_readfirstlane(wl + slot * G::WU + i * 1024)), "v"(off), "s"(base) : "memory");
    };

    // ---- scales
    int64_t srow[RT];                                              // element of the lane's row that its steps start at
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) srow[rt] = (int64_t)((row0 + rt * 16 < g.N ? row0 + rt * 16 : g.N - 16) + lr) * K;
    u32x2 win[RT], win_next[RT];                                   // windows of four steps (one that would pass the row's end starts earlier; kScDealt clamps step by step)
    const int row_steps = K >> 7;
    const auto load_window = [&](u32x2* dst, int s0) {
        if constexpr (SC == kScInt4Window) {
            const int c = c_begin + s0 < row_steps - 4 ? c_begin + s0 : row_steps - 4;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) dst[rt] = *(const u32x2_a1*)((const uint16_t*)g.scales + (srow[rt] >> 7) + c);
        } else if constexpr (SC == kScDealt) {
            const int c = c_begin + s0 + q < row_steps - 1 ? c_begin + s0 + q : row_steps - 1;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) dst[rt] = *(const u32x2_a1*)(g.scales + ((srow[rt] >> 7) + c) * 8);
        }
    };
    constexpr int SW = SC == kScUse ? 2 : 1;                       // scale words of a lane's 16 elements of a half step
    uint32_t sw[SC >= kScHalf ? RT : 1][SW], sw_next[SC >= kScHalf ? RT : 1][SW];
    const auto load_half = [&](int h_) {
        if constexpr (SC >= kScHalf) {
            const int h = h_ < halves ? h_ : halves - 1;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int i = 0; i < SW; ++i) {
                    const int64_t si = (srow[rt] + k_begin + h * 64 + q * 16 + i * 8) / g.group;
                    sw_next[rt][i] = g.scale_dtype == XQ_SCALE_F32 ? ((const uint32_t*)g.scales)[si] : (uint32_t)((const uint16_t*)g.scales)[si] << 16;
                }
        }
    };
    float ts[RT];                                                  // block-fp8: lane l holds the scale of step l
    if constexpr (SC == kScFp8) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const int n = row0 + rt * 16 < g.N ? row0 + rt * 16 : g.N - 16;
            const int c = c_begin + (lane < n_steps ? lane : n_steps - 1);
            ts[rt] = ((const float*)g.scales)[(int64_t)(n >> 7) * row_steps + (c > 0 ? c : 0)];
        }
    }
    const float gsc = FMT == XQ_FMT_NVFP4 ? g.global_scale[0] : 1.0f;
    const float* nf4_lds = (const float*)(smem + kStreamWaves * G::WAVE);
    if (FMT == XQ_FMT_NF4) {
        if (tid < 16) ((float*)(smem + kStreamWaves * G::WAVE))[tid] = kNf4Level[tid];
        __syncthreads();
    }

    f32x4 acc[RT][MT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[rt][mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    f32x4 su[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) su[mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // ---- the stream.  Nothing in it is shared between waves: a wave waits for its own loads by count.
    if (n_steps > 0) {
        load_window(win, 0);
        load_half(0);
        // First what the first products need -- the scales, x, half of the row tiles -- and a wait for it; then the others' weights, for
        // which the first half step waits when it comes to them, and the rest as if half steps before the first had asked for it.
        constexpr int P = XB > WB * HPW ? XB : WB * HPW;
#pragma unroll
        for (int i = 0; i < G::NX; ++i) issue_x1(0, 0, i);
#pragma unroll
        for (int i = 0; i < 2 * G::EARLY; ++i) issue_w1(0, 0, i);
        next_unit();
        if (su_step < n_steps) load_a();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {                          // (what the compiler waits for it waits for here)
            if constexpr (SC == kScFp8) asm volatile("" : "+v"(ts[rt]));
            else if constexpr (SC < kScHalf) asm volatile("" : "+v"(win[rt]));
            else asm volatile("" : "+v"(sw_next[rt][0]), "+v"(sw_next[rt][SW - 1]));
        }
#pragma unroll
        for (int i = 2 * G::EARLY; i < G::NW; ++i) issue_w1(0, 0, i);
#pragma unroll
        for (int v = -P; v < 0; ++v) {
            if (v + XB > 0)
#pragma unroll
                for (int i = 0; i < G::NX; ++i) issue_x1(v + XB, (v + XB) % XB, i);
            if (G::issues_w(v) && (v + 2) / HPW - 1 + WB > 0)
#pragma unroll
                for (int i = 0; i < G::NW; ++i) issue_w1((v + 2) / HPW - 1 + WB, ((v + 2) / HPW - 1 + WB) % WB, i);
        }
        const int x_lane = lr * 128, x_sw = (lr >> 1) & 5;
        int w_slot = 0, x_slot = 0, unit = 0;
        u32x4 w[RT][FMT == XQ_FMT_FP8 ? 2 : 1];
        const auto half_step = [&](auto hh_, auto odd_, int s, int ph) {
            constexpr int hh = decltype(hh_)::value, odd = decltype(odd_)::value;       // odd: the step's place in its unit
            constexpr bool LATE = hh == 0 && odd == 0 && G::EARLY < RT;                  // the later row tiles' weights are waited for on the way
            const int h = 2 * s + hh;
            constexpr int N = G::ahead(64 + 2 * odd + hh);
            if (hh || odd || s) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N < 63 ? N : 63) : "memory");
            bf16x8 xf[2][MT];
#pragma unroll
            for (int jj = 0; jj < 2; ++jj)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    xf[jj][mt] = *(const bf16x8*)(xs + x_slot * G::XH + mt * 2048 + x_lane + (((2 * q + jj) ^ x_sw) << 4));
            // the step's weights: block-fp8 piece 4 hh + q of a row (both half steps at once: the unit's slot is then free); 4-bit
            // piece 4 (step in the unit) + 2 hh + q / 2
            const auto read_w = [&](int rt) {
                const unsigned char* p = wsm + w_slot * G::WU + lr * 128 + rt * 2048;
                if constexpr (FMT == XQ_FMT_FP8) {
                    w[rt][0] = *(const u32x4*)(p + ((q ^ (lr >> 1)) << 4));
                    w[rt][1] = *(const u32x4*)(p + (((4 + q) ^ (lr >> 1)) << 4));
                } else {
                    const int c = 4 * odd + (q >> 1);
                    const u32x2 lo = *(const u32x2*)(p + ((c ^ (lr >> 1)) << 4) + (q & 1) * 8);
                    const u32x2 hi = *(const u32x2*)(p + (((c + 2) ^ (lr >> 1)) << 4) + (q & 1) * 8);
                    w[rt][0] = u32x4{lo[0], lo[1], hi[0], hi[1]};
                }
            };
            if constexpr (hh == 0) {
#pragma unroll
                for (int rt = 0; rt < (LATE ? G::EARLY : RT); ++rt) read_w(rt);
            }
            float s0[RT], s1[RT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                s1[rt] = 0.0f;
                if constexpr (SC == kScFp8) {
                    s0[rt] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ts[rt]), s));
                } else if constexpr (SC == kScInt4Window) {
                    const int c = c_begin + s - ph;
                    const int i = ph + (c < row_steps - 4 ? 0 : c - (row_steps - 4));          // uniform, 0 .. 3
                    const uint64_t v = (uint64_t)win[rt][1] << 32 | win[rt][0];
                    s0[rt] = __uint_as_float((uint32_t)(v >> (16 * i)) << 16);
                    s1[rt] = -8.0f * s0[rt];
                } else if constexpr (SC == kScDealt) {
                    const uint32_t v = (uint32_t)__builtin_amdgcn_ds_bpermute((ph * 16 + lr) * 4, (int)win[rt][hh]);
                    s0[rt] = FMT == XQ_FMT_NF4 ? __uint_as_float(v) : e4m3_to_f32((uint8_t)(v >> (8 * q))) * gsc;
                } else {
#pragma unroll
                    for (int i = 0; i < SW; ++i) sw[rt][i] = sw_next[rt][i];
                    s0[rt] = __uint_as_float(sw[rt][0]) * (FMT == XQ_FMT_NVFP4 ? gsc : 1.0f);
                    s1[rt] = -8.0f * s0[rt];
                }
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            load_half(h + 1);
            __builtin_amdgcn_sched_barrier(0);
            // the requests go out between the products, a few at a time: all at once they hold the wave up
            constexpr bool W = G::issues_w(2 * odd + hh);
            constexpr int LOADS = G::NX + (W ? G::NW : 0), SPREAD = (LOADS + 2 * RT - 1) / (2 * RT), EACH = SPREAD < 2 ? 2 : SPREAD;
            // (no weight is asked for before the late tiles have left the slot)
            constexpr int LX = (G::NX + 2 * G::EARLY - 1) / (2 * G::EARLY), SLOTS = 2 * (LATE ? RT - G::EARLY : RT), LW = (G::NW + SLOTS - 1) / SLOTS;
            const auto request = [&](int at) {                     // behind the at-th of the half step's 2 RT products
                if constexpr (LATE) {
#pragma unroll
                    for (int i = at * LX; i < (at + 1) * LX && i < G::NX; ++i) issue_x1(h + XB, x_slot, i);
                    if constexpr (W)
#pragma unroll
                        for (int i = (at - 2 * G::EARLY) * LW; i < (at - 2 * G::EARLY + 1) * LW && i < G::NW; ++i)
                            if (i >= 0) issue_w1(unit + WB, w_slot, i);
                } else {
#pragma unroll
                    for (int i = at * EACH; i < (at + 1) * EACH && i < LOADS; ++i) {
                        if (i < G::NX) issue_x1(h + XB, x_slot, i);
                        else issue_w1(unit + WB, w_slot, i - G::NX);
                    }
                }
            };
            // nf4: the levels of a product's codes, looked up while the product before is converted (two waves a SIMD do not hide the way
            // through LDS).  MLP forwards, us, each product's own lookups first and this: 4096/12288 24 rows 57.3 -> 53.6, 48 rows 63.4 -> 59.3,
            // 64 rows 70.8 -> 68.3, 4992/13056 3 rows r 64 72.1 -> 66.9.  Levels in a lane's register, by ds_bpermute (no LDS, four row tiles
            // of 16 rows pair): 64.9 at 24 rows, 76.4 at 64.  Those of the next half step's first product too: level.
            float level[2][8];
            const auto look_up = [&](int at) {
                if constexpr (FMT == XQ_FMT_NF4) {
                    uint32_t even = (w[at >> 1][0][2 * hh + (at & 1)] << 2) & 0x3c3c3c3cu, odd4 = (w[at >> 1][0][2 * hh + (at & 1)] >> 2) & 0x3c3c3c3cu;
                    asm volatile("" : "+v"(even), "+v"(odd4));      // (byte offsets of levels, a byte each: one instruction takes one out)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        level[at & 1][2 * i] = *(const float*)((const unsigned char*)nf4_lds + ((even >> (8 * i)) & 0xffu));
                        level[at & 1][2 * i + 1] = *(const float*)((const unsigned char*)nf4_lds + ((odd4 >> (8 * i)) & 0xffu));
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            look_up(0);
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                if constexpr (LATE) {
                    if (rt == G::EARLY) {
                        constexpr int OUT = G::NX + (G::spare() < G::behind_w() ? G::spare() : G::behind_w());
                        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(OUT < 63 ? OUT : 63) : "memory");
#pragma unroll
                        for (int t = G::EARLY; t < RT; ++t) read_w(t);
                        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                        look_up(2 * G::EARLY);
                    }
                }
#pragma unroll
                for (int jj = 0; jj < 2; ++jj) {
                    bf16x8 wf;
                    if (2 * rt + jj + 1 < 2 * RT && !(LATE && 2 * rt + jj + 1 == 2 * G::EARLY)) look_up(2 * rt + jj + 1);
                    if constexpr (FMT == XQ_FMT_NF4) {
                        const float* lv = level[jj];
                        wf = __builtin_bit_cast(bf16x8, u32x4{pack_bf16x2(lv[0] * s0[rt], lv[1] * s0[rt]), pack_bf16x2(lv[2] * s0[rt], lv[3] * s0[rt]),
                                                              pack_bf16x2(lv[4] * s0[rt], lv[5] * s0[rt]), pack_bf16x2(lv[6] * s0[rt], lv[7] * s0[rt])});
                    } else if constexpr (FMT == XQ_FMT_FP8) {
                        wf = decode8<FMT>(w[rt][hh][2 * jj], w[rt][hh][2 * jj + 1], s0[rt], 0.0f);
                    } else if constexpr (SC == kScUse) {
                        const float sv = __uint_as_float(sw[rt][jj]);
                        wf = decode8<FMT>(w[rt][0][2 * hh + jj], 0u, sv, -8.0f * sv);
                    } else {
                        wf = decode8<FMT>(w[rt][0][2 * hh + jj], 0u, s0[rt], s1[rt]);
                    }
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) acc[rt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xf[jj][mt], acc[rt][mt], 0, 0, 0);
                    request(2 * rt + jj);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            x_slot = x_slot + 1 == XB ? 0 : x_slot + 1;
            if constexpr (W) {
                ++unit;
                w_slot = w_slot + 1 == WB ? 0 : w_slot + 1;
            }
            if (s == su_step) {
#pragma unroll
                for (int jj = 0; jj < 2; ++jj)
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt)
                        su[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[2 * hh + jj]), xf[jj][mt], su[mt], 0, 0, 0);
                if (hh == 1) {
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) {
                        const int m = mt * 16 + lr;
                        if (m < M) *(f32x4*)(g.su_part + ((int64_t)(c_begin + s) * M + m) * g.r_pad + su_tile * 16 + q * 4) = su[mt];
                        su[mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                    }
                    next_unit();
                    if (su_step < n_steps) load_a();
                }
            }
        };
        using H0 = std::integral_constant<int, 0>;
        using H1 = std::integral_constant<int, 1>;
#pragma unroll 1
        for (int s0 = 0; s0 < n_steps; s0 += 4) {
            const int end = s0 + 4 < n_steps ? s0 + 4 : n_steps;
            if (RT <= 4 && end < n_steps) load_window(win_next, end);
#pragma unroll 1
            for (int s = s0; s < end; ++s) {
                half_step(H0{}, H0{}, s, s - s0);
                half_step(H1{}, H0{}, s, s - s0);
                if constexpr (HPW == 4) {
                    if (++s >= end) break;
                    half_step(H0{}, H1{}, s, s - s0);
                    half_step(H1{}, H1{}, s, s - s0);
                }
            }
            if constexpr (RT <= 4) {
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) win[rt] = win_next[rt];
            } else {
                if (end < n_steps) load_window(win, end);          // (no registers for two windows)
            }
        }
    }

    // ---- the eight waves' sums meet in LDS, GT row tiles at a time, and are added in wave order.  Lane (m = lr, quarter q) holds 4
    // consecutive weight rows of each row tile.
    constexpr int GT0 = G::WAVE / (MT * 1024), GT = GT0 < RT ? GT0 : RT;
    static_assert(GT >= 1, "the reduction needs room for a row tile");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    f32x4* red = (f32x4*)smem;
#pragma unroll
    for (int t0 = 0; t0 < RT; t0 += GT) {
        __syncthreads();
#pragma unroll
        for (int t = 0; t < GT; ++t)
            if (t0 + t < RT) {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) red[((wave * GT + t) * MT + mt) * 64 + lane] = acc[t0 + t][mt];
            }
        __syncthreads();
        for (int i = wave; i < GT * MT; i += kStreamWaves) {
            const int t = i / MT, mt = i - t * MT, m = mt * 16 + lr, n = row0 + (t0 + t) * 16;
            if (t0 + t < RT && n < g.N && rb * (16 * RT) < g.N) {   // uniform
                f32x4 v = red[i * 64 + lane];
#pragma unroll
                for (int w8 = 1; w8 < kStreamWaves; ++w8) v += red[(w8 * GT * MT + i) * 64 + lane];
                if (m < M) *(f32x4*)(g.partial + ((int64_t)split * M + m) * g.N + n + q * 4) = v;
            }
        }
    }
}

struct EpiJob {
    const float* partial;
    const float* su_part;
    const void* lora_B;        // [N, r] fp32 or bf16
    const bf16_t* bias;
    bf16_t* y;                 // GU: h, of the first job
    int64_t ldy;
    int32_t N, splits, parts, r, r_pad, lora_f32;
    float su_scale;
};
struct EpiBatch {
    EpiJob job[kStreamJobs];
};

// y[m][n..n+1] = sum_s part[s][m][n..] + bias + su_scale * sum_j su[m][j] * B[n][j], su = sum of the parts.  A wave takes 128
// columns (a lane 2) of RW rows, the block's waves the rows next to each other.  The kernel is a few dependent memory round
// trips long: everything it needs -- low-rank parts (dealt over all threads, met in LDS), partial tiles, B values of all ranks (NB
// chunks of 16) -- is requested before anything is waited for, in the order of use.  Every sum runs in a fixed order.
// NB: B's chunks were once fetched one behind the other, a trip to memory each: whole forwards at r 64, us, of 24 / 64 rows: int4
// [4096, 4096] 14.2 -> 13.6 / 17.0 -> 16.5, [7808, 2944] 15.6 -> 14.9 / 20.8 -> 20.0, fp8 [1024, 4096] 12.4 -> 11.8 / 14.6 -> 14.0; level at
// [12288, 4096] and r 16.
// RW: 1 up to 16 rows; above, 2 with eight splits requested at a time or 4 with four, by the rule in launch_skinny_stream.
// A block has four waves also where it has fewer than four rows: with a wave a row the pieces of B that so few threads would have
// taken were registers of every block, 368 for gate and up at r 64, one block a compute unit.  Whole forwards, us, before and now:
// MLP 4736/14208 1 row nf4 r 64 77.7 -> 66.1, 4608/12288 9 rows fp8 r 64 66.2 -> 57.9, 4992/14848 16 rows int4 r 64 72.8 -> 65.7, 4224/14208 2
// rows nvfp4 r 32 53.2 -> 50.8; one weight [2048, 4736] 1 row nf4 r 64 13.5 -> 10.8.
// VEC: B is fp32 with r % 4 == 0 (16-byte pieces).  GU: jobs 0 and 1 are gate and up, h is written.
template <int RW, int NB, bool VEC, bool GU>
__global__ void __launch_bounds__(256)
stream_epilogue_kernel(int32_t M, int32_t first1, int32_t first2, int32_t first3, EpiBatch b) {
    constexpr int NP = GU ? 2 : 1;
    __shared__ __attribute__((aligned(16))) float su[NP][4 * RW][64];
    __shared__ f32x4 red[NP][256];
    __shared__ f32x4 bt[NP][NB][512];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int bx = blockIdx.x;
    const int ji = GU ? 0 : (bx >= first1 ? 1 : 0) + (bx >= first2 ? 1 : 0) + (bx >= first3 ? 1 : 0);
    const int at = bx - (ji == 0 ? 0 : ji == 1 ? first1 : ji == 2 ? first2 : first3);
    const int m0 = blockIdx.y * (4 * RW);
    constexpr int nthreads = 256;
    const EpiJob& g0 = b.job[ji];
    const int n = at * 128 + lane * 2;
    const int nn = n < g0.N ? n : 0;                               // N % 2 == 0
    const int mw = m0 + wave * RW;

    // B values of 16 ranks of the block's columns: fetched in 16-byte pieces of 4 ranks, neighbouring threads on neighbouring
    // pieces, and shared through LDS; piece P = column * 4 + ranks / 4 lies at P ^ (column / 4 & 7), which lets the 16 lanes of a
    // read pass (two columns a lane) fall on 16 different pieces
    constexpr int kPieces = 512 / nthreads;                        // of a thread
    f32x4 bq[NP][NB][kPieces];
    const auto load_b = [&](int p, int rc) {
        const EpiJob& g = b.job[ji + p];
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const int P = tid + i * nthreads, col = at * 128 + (P >> 2), j = 16 * rc + 4 * (P & 3);
            const int64_t row = (int64_t)(col < g.N ? col : 0) * g.r;
            if constexpr (VEC) {
                bq[p][rc][i] = *(const f32x4*)((const float*)g.lora_B + row + (j < g.r ? j : 0));
            } else {
#pragma unroll
                for (int f = 0; f < 4; ++f) {
                    const int64_t bi = row + (j + f < g.r ? j + f : 0);
                    bq[p][rc][i][f] = g.lora_f32 ? ((const float*)g.lora_B)[bi] : bf16_to_f32(((const bf16_t*)g.lora_B)[bi]);
                }
            }
        }
    };
    const auto store_b = [&](int p, int rc) {
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const int P = tid + i * nthreads;
            bt[p][rc][P ^ ((P >> 4) & 7)] = bq[p][rc][i];
        }
    };
    constexpr int SB = RW == 2 ? 8 : 4;                            // splits requested at a time
    f32x2 t[NP][SB][RW];
    const auto load_part = [&](int p, int s0) {
        const EpiJob& g = b.job[ji + p];
        const int64_t ss = (int64_t)M * g.N;
#pragma unroll
        for (int v = 0; v < SB; ++v)
#pragma unroll
            for (int u = 0; u < RW; ++u)
                t[p][v][u] = *(const f32x2*)(g.partial + (int64_t)(s0 + v < g.splits ? s0 + v : g.splits - 1) * ss + (int64_t)(mw + u < M ? mw + u : M - 1) * g.N + nn);
    };
    // (in the order in which they are waited for)
    f32x4 sp[NP][8];
    const auto load_su = [&](int p, int p0) {                      // thread (quad of ranks of a row, group of parts)
        const EpiJob& g = b.job[ji + p];
        const int qr = g.r_pad >> 2, quads = 4 * RW * qr, groups = nthreads / quads;
        const int qd = tid % quads, gi = tid / quads, m = qd / qr;
        const float* src = g.su_part + (int64_t)(m0 + m < M ? m0 + m : M - 1) * g.r_pad + (qd - m * qr) * 4;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int pi = p0 + gi + u * groups;
            sp[p][u] = *(const f32x4*)(src + (int64_t)(pi < g.parts ? pi : g.parts - 1) * M * g.r_pad);
        }
    };
#pragma unroll
    for (int p = 0; p < NP; ++p)
        if (b.job[ji + p].r > 0) load_su(p, 0);
#pragma unroll
    for (int p = 0; p < NP; ++p) load_part(p, 0);
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int rc = 0; rc < NB; ++rc)
            if (16 * rc < b.job[ji + p].r) load_b(p, rc);

    // ---- su of the block's rows -> LDS
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const EpiJob& g = b.job[ji + p];
        if (g.r > 0) {
            const int quads = RW * g.r_pad, groups = nthreads / quads, gi = tid / quads;
            f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
            for (int p0 = 0;;) {
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (p0 + gi + u * groups < g.parts) v += sp[p][u];
                p0 += 8 * groups;
                if (p0 >= g.parts) break;
                load_su(p, p0);
            }
            red[p][tid] = v;
        }
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const EpiJob& g = b.job[ji + p];
        if (g.r > 0) {
            const int qr = g.r_pad >> 2, quads = 4 * RW * qr, groups = nthreads / quads;
            if (tid < quads) {
                f32x4 v = red[p][tid];
                for (int gi = 1; gi < groups; ++gi) v += red[p][gi * quads + tid];
                const int m = tid / qr, j = (tid - m * qr) * 4;
#pragma unroll
                for (int e = 0; e < 4; ++e) su[p][m][j + e] = j + e < g.r ? v[e] * g.su_scale : 0.0f;
            }
        }
    }
    f32x2 o[NP][RW];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const EpiJob& g = b.job[ji + p];
#pragma unroll
        for (int u = 0; u < RW; ++u) o[p][u] = f32x2{0.0f, 0.0f};
        for (int s0 = 0;;) {
#pragma unroll
            for (int v = 0; v < SB; ++v)
                if (s0 + v < g.splits) {
#pragma unroll
                    for (int u = 0; u < RW; ++u) {
                        o[p][u][0] += t[p][v][u][0];
                        o[p][u][1] += t[p][v][u][1];
                    }
                }
            s0 += SB;
            if (s0 >= g.splits) break;
            load_part(p, s0);
        }
    }
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int rc = 0; rc < NB; ++rc)
            if (16 * rc < b.job[ji + p].r) store_b(p, rc);
    __syncthreads();
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const EpiJob& g = b.job[ji + p];
#pragma unroll
        for (int rc = 0; rc < NB; ++rc) {
            if (16 * rc >= g.r) break;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                f32x4 bv[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) bv[e] = bt[p][rc][((lane * 2 + e) * 4 + c) ^ ((lane >> 1) & 7)];
#pragma unroll
                for (int u = 0; u < RW; ++u) {
                    const f32x4 sv = *(const f32x4*)&su[p][wave * RW + u][16 * rc + 4 * c];
#pragma unroll
                    for (int f = 0; f < 4; ++f)
#pragma unroll
                        for (int e = 0; e < 2; ++e) o[p][u][e] = __builtin_fmaf(sv[f], bv[e][f], o[p][u][e]);
                }
            }
        }
        if (g.bias) {
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const float bb = bf16_to_f32(g.bias[nn + e]);
#pragma unroll
                for (int u = 0; u < RW; ++u) o[p][u][e] += bb;
            }
        }
    }
    if (n >= g0.N) return;
#pragma unroll
    for (int u = 0; u < RW; ++u) {
        if (mw + u < M) {
            f32x2 r = o[0][u];
            if constexpr (GU) {
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const float gate = round_bf16(r[e]);
                    r[e] = round_bf16(gate * sigmoid_f32(gate)) * round_bf16(o[NP - 1][u][e]);
                }
            }
            *(uint32_t*)(g0.y + (int64_t)(mw + u) * g0.ldy + n) = pack_bf16x2(r[0], r[1]);
        }
    }
}

static inline int64_t al256(int64_t b) { return (b + 255) & ~(int64_t)255; }

// (the storages that xq_validate_weight and skinny_supported leave: nf4 fp32, nvfp4 e4m3 or fp32, int4 fp32 or bf16)
static int scale_mode(const xq_weight* w) {
    if (w->format == XQ_FMT_FP8) return kScFp8;
    if (w->format == XQ_FMT_NF4) return kScDealt;
    if (w->format == XQ_FMT_NVFP4) return w->scale_dtype == XQ_SCALE_E4M3 ? kScDealt : kScHalf;
    if (w->group == 128 && w->scale_dtype == XQ_SCALE_BF16) return kScInt4Window;
    return w->group % 16 == 0 && w->cols % w->group == 0 ? kScHalf : kScUse;
}

// ---- plans
// What the plans have to know of a storage: the row tiles of a block at most (the uncommon scale storages keep more registers per tile),
// the LDS it takes beside the waves' parts, the steps of a unit of its weights, and what a half step costs for each row tile, in us.
constexpr int row_tiles_max(int sc) { return sc >= kScHalf ? 2 : 8; }
enum { kPlan4Bit = 0, kPlanFp8 = 1, kPlanNf4 = 2, kPlanUncommon = 3, kPlanClasses = 4 };
static int plan_class(const xq_weight* w) {
    return scale_mode(w) >= kScHalf ? kPlanUncommon : w->format == XQ_FMT_FP8 ? kPlanFp8 : w->format == XQ_FMT_NF4 ? kPlanNf4 : kPlan4Bit;
}
struct PlanClass {
    int row_tiles, levels, unit;
    double row_us;
};
static const PlanClass kPlans[kPlanClasses] = {
    {row_tiles_max(kScInt4Window), 0, 2, 0.30}, {row_tiles_max(kScFp8), 0, 1, 0.20}, {row_tiles_max(kScDealt), stream_levels(XQ_FMT_NF4), 2, 0.36}, {row_tiles_max(kScHalf), 0, 2, 0.30}};

// The row tiles of a block that make a launch shortest by an estimate of what it takes beyond a constant, in us (they change nothing in
// the results); `tiles`, `splits` of each forward of the launch, `steps` of the longest split.  Rounds of the chip, and in a block the half
// steps of a wave, each for its weights, its x and their products; a second block on the compute unit nearly doubles them.
// Steps that leave a wave's last weight unit half empty cost more than they multiply.  The constants, and those of make_stream_splits,
// are the ones whose plans were shortest in a sweep of every (splits, row tiles) on 808 single forwards and 218 MLPs of 2 to 64 rows in all
// formats: 1.7 per cent behind the best of the sweep on average, singles 2.0, MLPs 0.3; constants that were fitted to the times themselves 2.3, 2.8
// and 0.7 (int4 [4352, 4352] of 64 rows 18.7 us with five splits of six row tiles where three of four take 15.7).  Where a tile of five or seven
// rows spares a round of the chip the whole forward is up to 11 per cent shorter (MLP 3712/9344 of 24 rows int4 46.3 -> 42.6, 4096/12416 of
// 24 rows int4 52.2 with four tiles, 48.6 with seven, nf4 66.0 -> 61.2).
static int stream_row_tiles(const int* tiles, const int* splits, int n, int steps, int mt, const PlanClass& c, double* us) {
    const int cus = num_cus(), wave_steps = (steps + kStreamWaves - 1) / kStreamWaves;
    const double halves = 2 * wave_steps + (wave_steps % c.unit ? 0.4 : 0);
    int best = 1;
    double least = 0;
    for (int rt = 1; rt <= c.row_tiles && stream_fits(c.levels, mt, rt); ++rt) {
        int blocks = 0;
        for (int i = 0; i < n; ++i) blocks += (tiles[i] + rt - 1) / rt * splits[i];
        const bool pair = stream_pairs(c.levels, mt, rt);
        const int per_cu = pair ? 2 : 1, rounds = (blocks + cus * per_cu - 1) / (cus * per_cu), on_cu = std::min((blocks + cus - 1) / cus, rounds * per_cu);
        const double half = c.row_us * rt + 0.25 * mt + 0.003 * rt * mt;
        const double t = rounds * ((pair ? 2.25 : 3.75) + 0.2 * rt + 0.16 * rt * mt + halves * half * (1.0 + 0.9 * ((double)on_cu / rounds - 1.0)));
        if (least == 0 || t < least) { least = t; best = rt; }
    }
    if (us) *us = least;
    return best;
}
// steps of a split at most (a lane holds one block-fp8 scale of a wave's steps)
constexpr int kStreamSteps = 64 * kStreamWaves;
static int least_stream_splits(int64_t K) { return (int)xq_cdiv(K >> 7, kStreamSteps); }
// splits that a plan may have: 64, sums of 16 MB, four steps in the longest.  Workspaces are sized for as many, whatever the storage: its plan
// would be two to five microseconds of a first call (all four classes at [1024, 4096] and [4096, 12288]), its memory a few MB less.
static int most_stream_splits(int64_t M, int64_t N, int64_t K) {
    return (int)std::max<int64_t>(least_stream_splits(K), std::min(std::min<int64_t>(64, (16ll << 20) / (M * N * 4)), ((K >> 7) - 1) / (kStreamWaves / 2 - 1)));
}
// K splits of a forward, by its own shape and storage: the cheapest sum of that and of the epilogue's share, 0.48 us a split and the partial
// sums' trip.  Weights twice as wide as deep are mostly gate and up of an MLP, whose one launch has other rounds than a weight alone: 0.55
// of what a pair takes counts too (nvfp4 4096 -> 2 x 12288 of 19 rows, the whole MLP: 49.4 us with two splits, 44.1 with one; alone they
// are level).
static int make_stream_splits(int cls, int64_t M, int64_t N, int64_t K) {
    const int ct = (int)(K >> 7), mt = (int)xq_cdiv(M, 16), most = most_stream_splits(M, N, K);
    const int tiles[2] = {(int)(N / 16), (int)(N / 16)};
    int best = 0, last_steps = 0;
    double best_cost = 0;
    for (int s = least_stream_splits(K); s <= most; ++s) {
        const int steps = (int)xq_cdiv(ct, s), splits[2] = {s, s};
        if (steps == last_steps) continue;                         // more splits, none of them shorter
        last_steps = steps;
        const double sums = s * (0.48 + M * N * 8 * 0.145e-6);
        double c, two = 0;
        stream_row_tiles(tiles, splits, 1, steps, mt, kPlans[cls], &c);
        c += sums;
        if (N >= 2 * K) {
            stream_row_tiles(tiles, splits, 2, steps, mt, kPlans[cls], &two);
            c += 0.55 * (two + 2 * sums);
        }
        if (best == 0 || c < best_cost) { best = s; best_cost = c; }
    }
    return best;
}

// splits, and the row tiles of a launch alone
struct StreamPlan {
    int splits, row_tiles;
};
static StreamPlan stream_plan(int cls, int64_t M, int64_t N, int64_t K) {
    static thread_local PlanSlot<StreamPlan> kept[64];
    const PlanKey key{M, N, K, num_cus(), cls};
    PlanSlot<StreamPlan>& e = kept[key.slot()];
    if (!(e.key == key)) {
        const int tiles = (int)(N / 16), splits = make_stream_splits(cls, M, N, K);
        e = PlanSlot<StreamPlan>{key, {splits, stream_row_tiles(&tiles, &splits, 1, (int)xq_cdiv(K >> 7, splits), (int)xq_cdiv(M, 16), kPlans[cls], nullptr)}};
    }
    return e.value;
}

// whether a forward of this shape runs on the two launches of this file (and not in one, xq_skinny_rows.hip)
bool skinny_takes_stream(const xq_weight* w, int64_t M, int64_t ldx, const void* lora_A, const void* lora_B, int lora_dtype, int r) {
    return skinny_supported(w, M) && stream_takes_pitch(M, ldx) && !(skinny_rows_enabled() && skinny_rows_supported(w, M, lora_A, lora_B, lora_dtype, r));
}

void skinny_stream_plan(const xq_weight* w, int64_t M, int32_t* plan) {
    const StreamPlan p = stream_plan(plan_class(w), M, w->rows, w->cols);
    plan[0] = p.splits;
    plan[1] = p.row_tiles;
}

int64_t skinny_workspace_bytes(int64_t M, int64_t N, int64_t K, int r_pad) {
    if (M < 1 || K < 128 || N < 16) return 256;
    const int rp = r_pad ? r_pad : 16;
    // (never less than a partial sum for every 32, 16 or 8 steps, whatever the plan: what callers have always been asked for)
    const int64_t s = most_stream_splits(M, N, K), held = xq_cdiv(K >> 7, M <= 16 ? 32 : M <= 32 ? 16 : 8);
    return al256((s > held ? s : held) * M * N * 4) + al256((K >> 7) * M * rp * 4) + 256;
}

bool skinny_supported(const xq_weight* w, int64_t M) {
    if (M < 1 || M > 64 || w->num_experts != 1) return false;
    if (w->format == XQ_FMT_NF4 && (w->group != 64 || w->scale_dtype != XQ_SCALE_F32)) return false;   // other nf4 storages take the tile kernels
    if (w->format != XQ_FMT_FP8 && w->layout != XQ_LAYOUT_FLAT) return false;
    if (w->cols % 128 != 0 || w->cols < 1024 || w->rows % 16 != 0) return false;
    if (w->format == XQ_FMT_INT4 && (w->group % 8 != 0)) return false;
    return true;
}

template <int FMT, int SC, int MT, int RT>
static int launch_stream_one(const StreamBatch& b, const int* first, const bf16_t* x, int64_t ldx, int64_t M, int64_t K, hipStream_t s) {
    constexpr int lds = kStreamWaves * StreamGeo<FMT, MT, RT>::WAVE + stream_levels(FMT);
    static_assert(lds <= 160 * 1024, "LDS of a block");
    static std::atomic<bool> attr_set{false};
    if (!attr_set) {
        const hipError_t e = hipFuncSetAttribute((const void*)stream_split_kernel<FMT, SC, MT, RT>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) {
            xq_set_error("xq_linear_fwd: cannot raise the dynamic LDS limit: %s", hipGetErrorString(e));
            return XQ_ERR_LAUNCH;
        }
        attr_set = true;
    }
    stream_split_kernel<FMT, SC, MT, RT><<<(unsigned)first[4], 64 * kStreamWaves, lds, s>>>(x, ldx, (int32_t)M, (int32_t)K, first[1], first[2], first[3], b);
    return XQ_OK;
}
template <int FMT, int SC, int MT>
static int launch_stream_mt(const StreamBatch& b, const int* first, const bf16_t* x, int64_t ldx, int64_t M, int64_t K, int rt, hipStream_t s) {
#define XQ_STREAM_TILES(RT)                                                            \
    if constexpr (RT <= row_tiles_max(SC) && stream_fits(stream_levels(FMT), MT, RT)) \
        if (rt == RT) return launch_stream_one<FMT, SC, MT, RT>(b, first, x, ldx, M, K, s)
    XQ_STREAM_TILES(1); XQ_STREAM_TILES(2); XQ_STREAM_TILES(3); XQ_STREAM_TILES(4);
    XQ_STREAM_TILES(5); XQ_STREAM_TILES(6); XQ_STREAM_TILES(7); XQ_STREAM_TILES(8);
#undef XQ_STREAM_TILES
    return XQ_ERR_UNSUPPORTED;
}
template <int FMT, int SC>
static int launch_stream_sc(const StreamBatch& b, const int* first, const bf16_t* x, int64_t ldx, int64_t M, int64_t K, int rt, hipStream_t s) {
    if (M <= 16) return launch_stream_mt<FMT, SC, 1>(b, first, x, ldx, M, K, rt, s);
    if (M <= 32) return launch_stream_mt<FMT, SC, 2>(b, first, x, ldx, M, K, rt, s);
    if (M <= 48) return launch_stream_mt<FMT, SC, 3>(b, first, x, ldx, M, K, rt, s);
    return launch_stream_mt<FMT, SC, 4>(b, first, x, ldx, M, K, rt, s);
}

bool skinny_stream_multi_supported(const SkinnyRowsJob* jobs, int n_jobs, int64_t M) {
    if (n_jobs < 1 || n_jobs > kStreamJobs) return false;
    for (int i = 0; i < n_jobs; ++i) {
        const xq_weight* w = jobs[i].w;
        if (!skinny_supported(w, M) || w->format != jobs[0].w->format || w->cols != jobs[0].w->cols ||
            scale_mode(w) != scale_mode(jobs[0].w) || !xq_aligned(w->packed, 16) || jobs[i].ldy % 4 != 0 || !xq_aligned(jobs[i].y, 8))
            return false;
        if (jobs[i].r > 0 && (!xq_aligned(jobs[i].lora_A, 16) || !xq_aligned(jobs[i].lora_B, 4))) return false;
    }
    return true;
}

int launch_skinny_stream(const SkinnyRowsJob* jobs, int n_jobs, bool swiglu, const bf16_t* x, int64_t ldx, int64_t M, int lora_dtype,
                         void* workspace, hipStream_t stream) {
    const xq_weight* w0 = jobs[0].w;
    const int64_t K = w0->cols;
    const int sc = scale_mode(w0), cls = plan_class(w0), mt = (int)xq_cdiv(M, 16);
    XQ_REQUIRE(stream_takes_pitch(M, ldx), "xq_linear_fwd: internal error: rows of x too far apart for the streaming kernel");
    StreamBatch b{};
    EpiBatch e{};
    uint8_t* ws = (uint8_t*)workspace;
    bool vec = true;
    int steps = 0, rt = 1;
    for (int i = 0; i < n_jobs; ++i) {
        const SkinnyRowsJob& j = jobs[i];
        const int rp = j.r > 0 ? (j.r + 15) / 16 * 16 : 0;
        const int64_t N = j.w->rows;
        StreamJob& g = b.job[i];
        const StreamPlan plan = stream_plan(cls, M, N, K);
        g.splits = plan.splits;
        rt = plan.row_tiles;
        g.packed = (const uint8_t*)j.w->packed; g.scales = (const uint8_t*)j.w->scales; g.global_scale = j.w->global_scale;
        g.N = (int)N; g.group = j.w->group; g.scale_dtype = j.w->scale_dtype;
        g.chunk_q = (int)(K >> 7) / g.splits; g.chunk_rem = (int)(K >> 7) % g.splits;
        const int longest = g.chunk_q + (g.chunk_rem ? 1 : 0);
        steps = longest > steps ? longest : steps;
        g.partial = (float*)ws;
        ws += al256((int64_t)g.splits * M * N * 4);
        g.su_part = (float*)ws;
        ws += al256((K >> 7) * M * (rp ? rp : 16) * 4) + 256;
        g.lora_A = rp ? j.lora_A : nullptr; g.lora_f32 = lora_dtype == XQ_DT_F32; g.r = j.r; g.r_pad = rp;
        EpiJob& ej = e.job[i];
        ej.partial = g.partial; ej.su_part = g.su_part; ej.lora_B = rp ? j.lora_B : nullptr; ej.bias = j.bias; ej.y = j.y; ej.ldy = j.ldy;
        ej.N = (int)N; ej.splits = g.splits; ej.parts = (int)(K >> 7); ej.r = j.r; ej.r_pad = rp; ej.lora_f32 = g.lora_f32; ej.su_scale = j.scaling;
        vec = vec && (j.r == 0 || (g.lora_f32 && j.r % 4 == 0 && xq_aligned(j.lora_B, 16)));
    }
    int tiles[kStreamJobs], splits[kStreamJobs];
    for (int i = 0; i < n_jobs; ++i) { tiles[i] = b.job[i].N / 16; splits[i] = b.job[i].splits; }
    if (n_jobs > 1) rt = stream_row_tiles(tiles, splits, n_jobs, steps, mt, kPlans[cls], nullptr);
    int first[5] = {0, 0, 0, 0, 0}, efirst[5] = {0, 0, 0, 0, 0};
    for (int i = 0; i < kStreamJobs; ++i) {
        first[i + 1] = first[i];
        efirst[i + 1] = efirst[i];
        if (i < n_jobs) {
            // (a weight of fewer row blocks than rank tiles gets blocks that only form a low-rank part)
            const int rank_tiles = b.job[i].r_pad >> 4, row_blocks = (int)xq_cdiv(tiles[i], (int64_t)rt);
            b.job[i].row_blocks = row_blocks > rank_tiles ? row_blocks : rank_tiles;
            first[i + 1] += b.job[i].row_blocks * b.job[i].splits;
            efirst[i + 1] += (int)xq_cdiv(b.job[i].N, 128);
        } else {
            b.job[i] = b.job[0];
            e.job[i] = e.job[0];
        }
    }
    int rc = XQ_ERR_UNSUPPORTED;
#define XQ_STREAM_CASE(F, S) \
    if (w0->format == F && sc == S) rc = launch_stream_sc<F, S>(b, first, x, ldx, M, K, rt, stream)
    XQ_STREAM_CASE(XQ_FMT_FP8, kScFp8);
    XQ_STREAM_CASE(XQ_FMT_INT4, kScInt4Window);
    XQ_STREAM_CASE(XQ_FMT_INT4, kScHalf);
    XQ_STREAM_CASE(XQ_FMT_INT4, kScUse);
    XQ_STREAM_CASE(XQ_FMT_NVFP4, kScDealt);
    XQ_STREAM_CASE(XQ_FMT_NVFP4, kScHalf);
    XQ_STREAM_CASE(XQ_FMT_NF4, kScDealt);
#undef XQ_STREAM_CASE
    if (rc) return rc;
    const unsigned cols = (unsigned)(swiglu ? efirst[1] : efirst[4]);
    // Four rows a wave and four splits at a time, us against two rows and eight (whole passes, all else equal):
    //  * two rows would be more than three blocks a compute unit: int4 [14720, 4864], 51 rows, r 32 / 64: 30.8 against 32.7 / 33.7 against
    //    36.1; MLP of 14720 x 4864, 64 rows: int4 94.0 / 99.7 and 104.4 / 111.8, nf4 109.4 / 114.8 and 120.5 / 127.6.  (At three blocks,
    //    12288 columns and 64 rows, four rows are level at r 16, 1.5 per cent slower at r 32, 3 at r 64; at 2.7, 14720 columns and 48
    //    rows, -3 to 1 per cent.)
    //  * no more than four splits, which are one request then: up to rank 16 (MLP of 9088 x 2944, 64 rows, nf4 51.4 against 52.8), to rank
    //    32 where a row of blocks fills half the chip ([16384, 2048], 17 rows 14.3 against 15.0); below that, and at r 64, two rows are up to
    //    4 per cent faster.
    //  * up to rank 16, where they are one block a compute unit and two rows a few blocks more than one: [5120, 1536], 64 rows 14.6
    //    against 15.3, [12288, 4096], 17 rows 18.7 against 19.2.
    int ranks = 0, most = 0;
    for (int i = 0; i < n_jobs; ++i) {
        ranks = e.job[i].r_pad > ranks ? e.job[i].r_pad : ranks;
        most = splits[i] > most ? splits[i] : most;
    }
    const int64_t by2 = xq_cdiv((int64_t)cols * xq_cdiv(M, 8), num_cus()), by4 = xq_cdiv((int64_t)cols * xq_cdiv(M, 16), num_cus());
    const bool four = by2 > 3 || (most <= 4 && ranks <= (2 * (int64_t)cols >= num_cus() ? 32 : 16)) || (ranks <= 16 && 17 * by4 < 10 * by2);
    const int rw = M <= 16 ? 1 : four ? 4 : 2;
    const dim3 grid(cols, (unsigned)xq_cdiv(M, 4 * rw));
#define XQ_EPI_NB(RW, NB)                                                                                                                      \
    do {                                                                                                                                       \
        if (swiglu) {                                                                                                                          \
            if (vec) stream_epilogue_kernel<RW, NB, true, true><<<grid, 256, 0, stream>>>((int)M, efirst[1], efirst[2], efirst[3], e);     \
            else stream_epilogue_kernel<RW, NB, false, true><<<grid, 256, 0, stream>>>((int)M, efirst[1], efirst[2], efirst[3], e);        \
        } else {                                                                                                                               \
            if (vec) stream_epilogue_kernel<RW, NB, true, false><<<grid, 256, 0, stream>>>((int)M, efirst[1], efirst[2], efirst[3], e);    \
            else stream_epilogue_kernel<RW, NB, false, false><<<grid, 256, 0, stream>>>((int)M, efirst[1], efirst[2], efirst[3], e);       \
        }                                                                                                                                      \
    } while (0)
#define XQ_EPI(RW)                       \
    do {                                 \
        if (ranks <= 16) XQ_EPI_NB(RW, 1); \
        else if (ranks <= 32) XQ_EPI_NB(RW, 2); \
        else XQ_EPI_NB(RW, 4);           \
    } while (0)
    if (rw == 1) XQ_EPI(1);
    else if (rw == 2) XQ_EPI(2);
    else XQ_EPI(4);
#undef XQ_EPI
#undef XQ_EPI_NB
    return XQ_OK;
}

// XQ_SKINNY_ROWS=0 (or xq_set_skinny_one_launch(0)) keeps every skinny forward on the two-launch organisation: a process-wide
// test switch, to be set while no other thread is inside the library
static int g_skinny_rows = [] { const char* e = getenv("XQ_SKINNY_ROWS"); return e ? atoi(e) : 1; }();
void set_skinny_rows(int enabled) { g_skinny_rows = enabled; }
bool skinny_rows_enabled() { return g_skinny_rows != 0; }

int launch_skinny(const xq_weight* w, const bf16_t* x, int64_t ldx, int64_t M, const void* lora_A, const void* lora_B,
                  int lora_dtype, int r, float scaling, const bf16_t* bias, bf16_t* y, int64_t ldy, void* workspace,
                  int64_t workspace_bytes, hipStream_t stream) {
    const int64_t N = w->rows, K = w->cols;
    const int rp = r <= 0 ? 0 : ((r + 15) / 16) * 16;
    XQ_REQUIRE(workspace && xq_aligned(workspace, 256) && workspace_bytes >= skinny_workspace_bytes(M, N, K, rp),
               "xq_linear_fwd: workspace missing, misaligned or too small for the skinny path");
    XQ_REQUIRE(ldx % 8 == 0 && xq_aligned(x, 16) && xq_aligned(w->packed, 16), "xq_linear_fwd: operands must be 16-byte aligned");
    XQ_REQUIRE(ldy % 4 == 0 && xq_aligned(y, 8), "xq_linear_fwd: output rows must be 8-byte aligned");
    XQ_REQUIRE(rp == 0 || (xq_aligned(lora_A, 16) && xq_aligned(lora_B, 4)), "xq_linear_fwd: lora_A must be 16-byte and lora_B 4-byte aligned");
    // algorithmic bytes: packed weight + scales + x + y (+ LoRA factors), for the roofline figure; the timed
    // region is the whole forward (both launches)
    const double wbytes = (double)xq_packed_bytes_per_expert(w) + (double)xq_scale_bytes_per_expert(w);
    const bool timed = xq_profile_mark_begin(stream, wbytes + 2.0 * M * K + 2.0 * M * N + 4.0 * r * (K + N));
    // M <= 16: one launch, whole rows per block, where the shape and the LoRA operands fit it and a slot is free (XQ_ERR_UNSUPPORTED: none
    // is, and the rows of x lie too far apart for the streaming kernels; nothing was launched)
    int rc = XQ_ERR_UNSUPPORTED;
    if (g_skinny_rows && skinny_rows_supported(w, M, lora_A, lora_B, lora_dtype, r))
        rc = launch_skinny_rows(w, x, ldx, M, lora_A, lora_B, r, scaling, bias, y, ldy, workspace, stream);
    if (rc == XQ_ERR_UNSUPPORTED && stream_takes_pitch(M, ldx)) {
        const SkinnyRowsJob job{w, lora_A, lora_B, rp ? r : 0, scaling, bias, y, ldy};
        rc = launch_skinny_stream(&job, 1, false, x, ldx, M, lora_dtype, workspace, stream);
    }
    if (timed) xq_profile_mark_end(stream);
    if (rc) return rc;
    XQ_CHECK_LAUNCH("skinny forward");
    return XQ_OK;
}

}  // namespace xq
