// Skinny-M (M <= 64) fused dequant-GEMM forward: the HBM-bound decode/rollout regime.
//
//   y[M, N] = x[M, K] . deq(W)^T + bias + s * (x . A^T) . B^T          (W FLAT [N, K])
//
// Every byte of the packed weight is read from HBM exactly once, decoded in registers to the exact bf16 value of the
// reference decoder and fed to v_mfma_f32_16x16x32_bf16 against x fragments.  Two launches for up to four forwards on one x
// (q + k + v, gate + up), no atomics, no zeroed buffers, fixed summation orders (deterministic):
//
//  1. stream_split_kernel: a grid of (row block) x (K split) tiles, one block of 8 waves per compute unit (two at M <= 32).
//     A wave owns 16 RT weight rows and streams them straight from memory into registers in the MFMA operand layout (a load
//     instruction takes 64 contiguous bytes of each of 16 rows), D steps of 128 elements in flight; rows are not shared
//     between waves, so the weight never passes through LDS.  x does: the block's whole slice [16 MT rows][K range] comes by
//     direct-to-LDS loads at the start (one barrier) and every wave reads its fragments from there -- the slice costs
//     1 / (8 RT) of what it would if each 16 weight rows fetched it, and nothing in the stream waits for a barrier.
//     The tile's sides balance what a block moves beside its weights, x (2 M K_b bytes) and fp32 partial sums
//     (8 M R_b bytes, written and read back): few, tall blocks for wide weights.  The blocks of `splits` leading tiles
//     compute the low-rank parts x . A^T of one split each.
//  2. stream_epilogue_kernel: sums the splits in order, adds bias and s * su . B^T in fp32 and rounds once to bf16; for gate
//     and up of an MLP it writes h = SwiGLU(gate, up) of the two rounded outputs instead.
//
// The split of K depends on a forward's own shape only: a joint launch gives the bits of the separate ones.
//
// What bounds it: at 64 rows the vector units (the 25 instructions that decode and feed one fragment of 8 weights a lane) and the
// matrix units, not memory: gate | up of 4096 -> 2 x 12288 in int4 takes 26 us (30 MB fetched) and its epilogue 13 us, half of
// which is the trip of the partial sums; at few rows the fixed costs of two dependent launches.  Forward of a SwiGLU MLP, us,
// against one that fetched x per 16 weight rows and ran gate, up, SwiGLU and down as separate launches:
//     int4  4096/12288, r 16: M = 24 62 -> 49, M = 64 90 -> 65      int4  2944/7808, r 32: M = 1 64 -> 34, M = 64 70 -> 49
//     fp8   4096/12288, r 16: M = 64 92 -> 76                       nvfp4 2944/7808, r 32: M = 1 71 -> 36
#include <stdlib.h>

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

// how a lane gets the scales of its codes: with the step's weights (one or two words), four steps' bf16 scales of int4
// groups of 128 in one load, four steps' 8 scale bytes dealt over the row's four lanes, per fragment at use, or (block-fp8)
// one value per row tile and step from registers
enum { kScFp8 = 0, kScInt4Window = 1, kScDealt = 2, kScStep = 3, kScUse = 4 };

// scales lie where their elements may: a pair of words from any byte (one global_load_dwordx2 like an aligned one)
typedef u32x2 u32x2_a1 __attribute__((aligned(1)));

// element offset of fragment (j, q) within a 128-element step: what lane q of a row holds after its loads (block-fp8: two
// loads of 16 bytes, 64 apart; 4-bit: one load of 16 bytes), so that a load instruction covers 64 contiguous bytes of a row
template <int FMT>
__device__ __forceinline__ int frag_k(int j, int q) {
    return FMT == XQ_FMT_FP8 ? (j >> 1) * 64 + q * 16 + (j & 1) * 8 : q * 32 + j * 8;
}

template <int FMT, int SC, int MT, int RT>
__global__ void __launch_bounds__(64 * kStreamWaves, MT == 4 || RT == 3 ? 2 : 4)
stream_split_kernel(const bf16_t* x, int32_t ldx, int32_t M, int32_t K, int32_t first1, int32_t first2, int32_t first3, StreamBatch b) {
    constexpr int EB = FMT == XQ_FMT_FP8 ? 1 : 2;                 // elements per byte
    constexpr int NL = FMT == XQ_FMT_FP8 ? 2 : 1;                 // 16-byte loads per lane, row tile and step
    constexpr int D = FMT == XQ_FMT_FP8 && RT > 1 ? 2 : 4;        // steps in flight
    constexpr int NS = SC != kScStep ? 0 : FMT == XQ_FMT_NVFP4 ? 2 : 1;   // scale words per row tile that travel with a step
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, lr = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int bx = blockIdx.x;
    const int ji = (bx >= first1 ? 1 : 0) + (bx >= first2 ? 1 : 0) + (bx >= first3 ? 1 : 0);
    const StreamJob& g = b.job[ji];
    const int at = bx - (ji == 0 ? 0 : ji == 1 ? first1 : ji == 2 ? first2 : first3);
    const int split = at % g.splits, rb = at / g.splits;
    const int c_begin = split * g.chunk_q + (split < g.chunk_rem ? split : g.chunk_rem);
    const int n_steps = g.chunk_q + (split < g.chunk_rem ? 1 : 0);
    const int k_begin = c_begin << 7;

    // ---- x slice -> LDS: [step][16 MT rows][16 pieces of 8 elements].  Piece (j, q) of row m lies at (4 j + q) ^ (m & 15): the
    // 16 lanes that one LDS pass of a fragment read serves fall on 16 different pieces.  Lane l of a load instruction lands at
    // piece l % 16 of row l / 16 of its four rows, so the swizzle is applied to the address it fetches.  (rows past M repeat the
    // last one: their products are never stored)
    {
        const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
        const int total = n_steps * MT * 4;
        for (int i = wave; i < total; i += kStreamWaves) {
            const int step = i / (MT * 4), m = (i % (MT * 4)) * 4 + (lane >> 4);
            const int col = (lane & 15) ^ (m & 15);
            const bf16_t* src = x + (int64_t)(m < M ? m : M - 1) * ldx + k_begin + step * 128 + frag_k<FMT>(col >> 2, col & 3);
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                         :: "s"(__builtin_amdgcn_readfirstlane(lds0 + i * 1024)), "v"(src) : "memory");
        }
    }
    // fragment (m tile, j) of step s: row lr of the tile
    int xo[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) xo[j] = lr * 256 + (((4 * j + q) ^ lr) << 4);
    const auto x_frag = [&](int s, int mt, int j) {
        return *(const bf16x8*)(smem + (s * MT + mt) * 4096 + xo[j]);
    };

    // ---- the low-rank parts: units of (step, 16 ranks) dealt over the waves of the split's blocks, the first of them over the
    // blocks.  A wave's first unit is requested here, behind the x slice and ahead of the weights, and multiplied before the
    // stream starts; D[rank][m] of one step goes out as it is (ranks >= r: whatever row 0 gives, never read).
    const int rank_tiles = g.r_pad >> 4, units = n_steps * rank_tiles, unit0 = rb + g.row_blocks * wave;
    const auto unit_base = [&](int u, int us) {
        const int row = (u - us * rank_tiles) * 16 + lr;
        return (int64_t)(row < g.r ? row : 0) * K + k_begin + us * 128;
    };
    const auto multiply_unit = [&](int u, int us, const u32x4 (&a)[4]) {
        const int jt = u - us * rank_tiles;
        f32x4 sacc[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) sacc[mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                sacc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[j]), x_frag(us, mt, j), sacc[mt], 0, 0, 0);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int m = mt * 16 + lr;
            if (m < M) *(f32x4*)(g.su_part + ((int64_t)(c_begin + us) * M + m) * g.r_pad + jt * 16 + q * 4) = sacc[mt];
        }
    };
    f32x4 araw[8];                                                 // fp32 factors (bf16 ones are not requested ahead)
    const auto load_unit = [&](int u) {
        const float* p = (const float*)g.lora_A + unit_base(u, u / rank_tiles);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            araw[2 * j] = *(const f32x4*)(p + frag_k<FMT>(j, q));
            araw[2 * j + 1] = *(const f32x4*)(p + frag_k<FMT>(j, q) + 4);
        }
    };
    if (g.lora_f32 && unit0 < units) load_unit(unit0);

    // ---- this wave's rows: tiles of 16 (N % 16 == 0: a tile is all in or all out; one past the end repeats the last)
    const int row0 = (rb * kStreamWaves + wave) * (16 * RT);
    const uint8_t* wp[RT];
    int64_t srow[RT];                                              // SC-dependent: the row's scales
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int n = (row0 + rt * 16 < g.N ? row0 + rt * 16 : g.N - 16) + lr;
        wp[rt] = g.packed + ((int64_t)n * K + k_begin) / EB + q * 16;
        srow[rt] = (int64_t)n * K + k_begin;
    }
    u32x4 w[D][RT][NL];
    uint32_t sw[D][RT][NS > 0 ? NS : 1];
    const auto load_step = [&](int slot, int s_) {
        const int s = s_ < n_steps ? s_ : n_steps - 1;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
            for (int i = 0; i < NL; ++i) w[slot][rt][i] = *(const u32x4*)(wp[rt] + (int64_t)s * (128 / EB) + i * 64);
            if constexpr (SC == kScStep && FMT == XQ_FMT_NVFP4) {
                const u32x2 v = *(const u32x2_a1*)((const uint32_t*)g.scales + ((srow[rt] + s * 128 + q * 32) >> 4));
                sw[slot][rt][0] = v[0];
                sw[slot][rt][1] = v[1];
            } else if constexpr (SC == kScStep) {
                const int64_t si = (srow[rt] + s * 128 + q * 32) / g.group;
                sw[slot][rt][0] = g.scale_dtype == XQ_SCALE_F32 ? ((const uint32_t*)g.scales)[si] : (uint32_t)((const uint16_t*)g.scales)[si] << 16;
            }
        }
    };
    // windows of four steps (a window that would pass the row's end starts earlier; kScDealt clamps step by step)
    u32x2 win[RT], win_next[RT];
    const int row_steps = K >> 7;
    const auto load_window = [&](u32x2* dst, int s0) {
        if constexpr (SC == kScInt4Window) {
            const int c = c_begin + s0 < row_steps - 4 ? c_begin + s0 : row_steps - 4;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
                dst[rt] = *(const u32x2_a1*)((const uint16_t*)g.scales + ((srow[rt] - k_begin) >> 7) + c);
        } else if constexpr (SC == kScDealt) {
            const int c = c_begin + s0 + q < row_steps - 1 ? c_begin + s0 + q : row_steps - 1;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) dst[rt] = *(const u32x2_a1*)(g.scales + ((srow[rt] - k_begin) >> 7) * 8 + (int64_t)c * 8);
        }
    };
    float ts[RT];                                                  // block-fp8: lane l holds the scale of step l
    if constexpr (SC == kScFp8) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const int n = row0 + rt * 16 < g.N ? row0 + rt * 16 : g.N - 16;
            ts[rt] = ((const float*)g.scales)[(int64_t)(n >> 7) * ((K + 127) >> 7) + c_begin + (lane < n_steps ? lane : n_steps - 1)];
        }
    }
    load_window(win, 0);
#pragma unroll
    for (int d = 0; d < D; ++d) load_step(d, d);
    const float gsc = FMT == XQ_FMT_NVFP4 ? g.global_scale[0] : 1.0f;
    float* nf4_lds = (float*)(smem + n_steps * MT * 4096);
    if (FMT == XQ_FMT_NF4 && tid < 16) nf4_lds[tid] = kNf4Level[tid];

    // the x slice is older than every load above: it has landed when no more than those are outstanding
    constexpr int kAhead = D * RT * (NL + (NS ? 1 : 0));
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kAhead < 63 ? kAhead : 63) : "memory");
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (g.lora_f32) {
#pragma unroll 1
        for (int u = unit0; u < units; u += g.row_blocks * kStreamWaves) {      // (more than one only for narrow weights of high rank)
            if (u != unit0) load_unit(u);
            u32x4 a[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                a[j] = u32x4{pack_bf16x2(araw[2 * j][0], araw[2 * j][1]), pack_bf16x2(araw[2 * j][2], araw[2 * j][3]),
                             pack_bf16x2(araw[2 * j + 1][0], araw[2 * j + 1][1]), pack_bf16x2(araw[2 * j + 1][2], araw[2 * j + 1][3])};
            multiply_unit(u, u / rank_tiles, a);
        }
    } else {
#pragma unroll 1
        for (int u = unit0; u < units; u += g.row_blocks * kStreamWaves) {
            const bf16_t* p = (const bf16_t*)g.lora_A + unit_base(u, u / rank_tiles);
            u32x4 a[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) a[j] = *(const u32x4*)(p + frag_k<FMT>(j, q));
            multiply_unit(u, u / rank_tiles, a);
        }
    }

    f32x4 acc[RT][MT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[rt][mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t sx[SC == kScDealt ? RT : 1][4];
    // register k of lane row r <- what lane row k fetched for lane row r
    const auto deal = [&]() {
        if constexpr (SC == kScDealt) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const u32x2 d = win[rt];
                const uint32_t x0 = d[0], x1 = FMT == XQ_FMT_NF4 ? d[0] : d[0] >> 16, x2 = d[1], x3 = FMT == XQ_FMT_NF4 ? d[1] : d[1] >> 16;
                const auto p02 = __builtin_amdgcn_permlane32_swap(x0, x2, false, false);
                const auto p13 = __builtin_amdgcn_permlane32_swap(x1, x3, false, false);
                const auto q01 = __builtin_amdgcn_permlane16_swap(p02[0], p13[0], false, false);
                const auto q23 = __builtin_amdgcn_permlane16_swap(p02[1], p13[1], false, false);
                sx[rt][0] = q01[0]; sx[rt][1] = q01[1]; sx[rt][2] = q23[0]; sx[rt][3] = q23[1];
            }
        }
    };
    const auto multiply = [&](int slot, int s, int ph) {              // ph: the step's place in its window
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
            } else if constexpr (SC == kScDealt && FMT == XQ_FMT_NF4) {
                s0[rt] = __uint_as_float(sx[rt][ph]);
            } else if constexpr (SC == kScDealt) {
                s0[rt] = e4m3_to_f32((uint8_t)sx[rt][ph]) * gsc;
                s1[rt] = e4m3_to_f32((uint8_t)(sx[rt][ph] >> 8)) * gsc;
            } else if constexpr (SC == kScStep && FMT == XQ_FMT_NVFP4) {
                s0[rt] = __uint_as_float(sw[slot][rt][0]) * gsc;
                s1[rt] = __uint_as_float(sw[slot][rt][NS > 1 ? 1 : 0]) * gsc;
            } else if constexpr (SC == kScStep) {
                s0[rt] = __uint_as_float(sw[slot][rt][0]);
                s1[rt] = -8.0f * s0[rt];
            }
        }
        bf16x8 xf[2][MT];                                          // fragments are read one j ahead
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) xf[0][mt] = x_frag(s, mt, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (j < 3) {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) xf[(j + 1) & 1][mt] = x_frag(s, mt, j + 1);
            }
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                bf16x8 wf;
                if constexpr (FMT == XQ_FMT_FP8) {
                    const u32x4 v = w[slot][rt][j >> 1];
                    wf = decode8<FMT>(v[2 * (j & 1)], v[2 * (j & 1) + 1], s0[rt], 0.0f);
                } else if constexpr (FMT == XQ_FMT_NVFP4) {
                    wf = decode8<FMT>(w[slot][rt][0][j], 0u, j < 2 ? s0[rt] : s1[rt], 0.0f);
                } else if constexpr (SC == kScUse) {
                    const float sv = load_scale(g.scales, (srow[rt] + s * 128 + q * 32 + j * 8) / g.group, g.scale_dtype);
                    wf = decode8<FMT>(w[slot][rt][0][j], 0u, sv, -8.0f * sv);
                } else {
                    wf = decode8<FMT>(w[slot][rt][0][j], 0u, s0[rt], s1[rt], nf4_lds);
                }
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) acc[rt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xf[j & 1][mt], acc[rt][mt], 0, 0, 0);
            }
        }
    };

    // ---- the stream: whole groups of four steps, each step's registers requested again once it has been multiplied, then the
    // remaining steps from what is in flight.  No branch lies between a load and its use, so every wait counts exactly.
    int s = 0;
#pragma unroll 1
    for (; s + 4 <= n_steps; s += 4) {
        deal();
        load_window(win_next, s + 4);
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            multiply(d % D, s + d, d);
            // (left alone the compiler decodes ahead, collects the products at the end and requests late)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) asm volatile("" : "+v"(acc[rt][mt]));
            load_step(d % D, s + d + D);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (SC == kScInt4Window || SC == kScDealt) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) win[rt] = win_next[rt];
        }
    }
    if (s < n_steps) {
        deal();
        multiply(0, s, 0);
        if constexpr (D == 2) load_step(0, s + 2);
        if (s + 1 < n_steps) multiply(1, s + 1, 1);
        if (s + 2 < n_steps) multiply(2 % D, s + 2, 2);
    }

    // ---- fp32 partial tile: lane (m = lr, quarter q) holds 4 consecutive weight rows of each row tile
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int n = row0 + rt * 16;
        if (n < g.N) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const int m = mt * 16 + lr;
                if (m < M) *(f32x4*)(g.partial + ((int64_t)split * M + m) * g.N + n + q * 4) = acc[rt][mt];
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
// trips long: everything the first sums need -- B values of the first 16 ranks, partial tiles, low-rank parts (dealt over all
// threads, met in LDS) -- is requested before anything is waited for.  Every sum runs in a fixed order.
// RW: 1 up to 16 rows; 2 with eight splits requested at a time above, against 4 rows and four splits, which took fewer blocks and
// twice the trips.  Whole forwards at r 16 / 64, us, of 24 rows: int4 [1024, 4096] 14.4 -> 12.4 / 18.8 -> 14.7, [4096, 4096] 15.1 -> 14.0 /
// 19.4 -> 16.3, [4096, 12288] 19.0 -> 17.5 / 26.9 -> 21.7; of 64 rows: 13.5 -> 12.5 / 18.1 -> 15.1, 15.9 -> 15.7 / 20.2 -> 18.2, 24.4 -> 23.4 /
// 32.1 -> 27.6.  [12288, 4096], where the epilogue is the smaller part, is level at r 16.
// VEC: B is fp32 with r % 4 == 0 (16-byte pieces).  GU: jobs 0 and 1 are gate and up, h is written.
template <int RW, bool VEC, bool GU>
__global__ void __launch_bounds__(256)
stream_epilogue_kernel(int32_t M, int32_t first1, int32_t first2, int32_t first3, EpiBatch b) {
    constexpr int NP = GU ? 2 : 1;
    __shared__ __attribute__((aligned(16))) float su[NP][4 * RW][64];
    __shared__ f32x4 red[NP][256];
    __shared__ f32x4 bt[NP][512];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int bx = blockIdx.x;
    const int ji = GU ? 0 : (bx >= first1 ? 1 : 0) + (bx >= first2 ? 1 : 0) + (bx >= first3 ? 1 : 0);
    const int at = bx - (ji == 0 ? 0 : ji == 1 ? first1 : ji == 2 ? first2 : first3);
    const int m0 = blockIdx.y * (4 * RW);
    const int nthreads = blockDim.x;
    const EpiJob& g0 = b.job[ji];
    const int n = at * 128 + lane * 2;
    const int nn = n < g0.N ? n : 0;                               // N % 2 == 0
    const int mw = m0 + wave * RW;

    // B values of 16 ranks of the block's columns: fetched in 16-byte pieces of 4 ranks, neighbouring threads on neighbouring
    // pieces, and shared through LDS; piece P = column * 4 + ranks / 4 lies at P ^ (column / 4 & 7), which lets the 16 lanes of a
    // read pass (two columns a lane) fall on 16 different pieces
    constexpr int kPieces = RW == 1 ? 8 : 2;                       // of a thread (RW > 1: always four waves)
    f32x4 bq[NP][kPieces];
    const auto load_b = [&](int p, int rc) {
        const EpiJob& g = b.job[ji + p];
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            if (i * nthreads < 512) {
                const int P = (tid + i * nthreads) & 511, col = at * 128 + (P >> 2), j = rc + 4 * (P & 3);
                const int64_t row = (int64_t)(col < g.N ? col : 0) * g.r;
                if constexpr (VEC) {
                    bq[p][i] = *(const f32x4*)((const float*)g.lora_B + row + (j < g.r ? j : 0));
                } else {
#pragma unroll
                    for (int f = 0; f < 4; ++f) {
                        const int64_t bi = row + (j + f < g.r ? j + f : 0);
                        bq[p][i][f] = g.lora_f32 ? ((const float*)g.lora_B)[bi] : bf16_to_f32(((const bf16_t*)g.lora_B)[bi]);
                    }
                }
            }
        }
    };
    const auto store_b = [&](int p) {
#pragma unroll
        for (int i = 0; i < kPieces; ++i)
            if (i * nthreads < 512) {
                const int P = (tid + i * nthreads) & 511;
                bt[p][P ^ ((P >> 4) & 7)] = bq[p][i];
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
#pragma unroll
    for (int p = 0; p < NP; ++p)
        if (b.job[ji + p].r > 0) load_b(p, 0);
#pragma unroll
    for (int p = 0; p < NP; ++p) load_part(p, 0);

    // ---- su of the block's rows -> LDS: thread (quad of ranks of a row, group of parts)
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const EpiJob& g = b.job[ji + p];
        if (g.r > 0) {
            const int qr = g.r_pad >> 2, quads = 4 * RW * qr, groups = nthreads / quads;
            const int qd = tid % quads, gi = tid / quads, m = qd / qr;
            const float* sp = g.su_part + (int64_t)(m0 + m < M ? m0 + m : M - 1) * g.r_pad + (qd - m * qr) * 4;
            f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
            for (int p0 = gi; p0 < g.parts; p0 += 8 * groups) {
                f32x4 a[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int pi = p0 + u * groups;
                    a[u] = *(const f32x4*)(sp + (int64_t)(pi < g.parts ? pi : g.parts - 1) * M * g.r_pad);
                }
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (p0 + u * groups < g.parts) v += a[u];
            }
            red[p][tid] = v;
            store_b(p);
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
    __syncthreads();
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const EpiJob& g = b.job[ji + p];
        for (int rc = 0; rc < g.r; rc += 16) {
            if (rc + 16 < g.r) load_b(p, rc + 16);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                f32x4 bv[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) bv[e] = bt[p][((lane * 2 + e) * 4 + c) ^ ((lane >> 1) & 7)];
#pragma unroll
                for (int u = 0; u < RW; ++u) {
                    const f32x4 sv = *(const f32x4*)&su[p][wave * RW + u][rc + 4 * c];
#pragma unroll
                    for (int f = 0; f < 4; ++f)
#pragma unroll
                        for (int e = 0; e < 2; ++e) o[p][u][e] = __builtin_fmaf(sv[f], bv[e][f], o[p][u][e]);
                }
            }
            if (rc + 16 < g.r) {
                __syncthreads();
                store_b(p);
                __syncthreads();
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

// What a launch of `blocks` blocks of 8 waves with RT row tiles and `steps` steps takes, in us, from a sweep of M 1..64 and widths
// 1024..16384: a start of ~4 us (launch, the x slice, the first weights), then the decode and the products of a SIMD's
// (row tile, step) units, which two waves to a SIMD overlap worse than four.  Two blocks are resident per CU at M <= 32, where
// their x slices fit.
static double stream_run_us(int64_t blocks, int rt, int steps, int mt) {
    const int per_cu = mt == 4 || rt == 3 || steps * mt * 4096 > 78 * 1024 ? 1 : 2;
    const int64_t cus = num_cus();
    const double rounds = (double)xq_cdiv(blocks, cus * per_cu);
    const double on_cu = (double)xq_cdiv(blocks, cus) < rounds * per_cu ? (double)xq_cdiv(blocks, cus) : rounds * per_cu;
    const double unit = on_cu > 1 && per_cu == 2 ? 0.12 + 0.04 * mt : 0.2 + 0.07 * mt;
    return 4.0 * rounds + on_cu * 2 * rt * steps * unit;
}
// row tiles of a wave by that estimate (they change nothing in the results); `tiles`, `splits` of each forward of the launch
static int stream_row_tiles(const int* tiles, const int* splits, int n, int steps, int mt, int rt_max, double* us) {
    int best = 1;
    double cost = 0;
    for (int rt = 1; rt <= rt_max; ++rt) {
        int64_t blocks = 0;
        for (int i = 0; i < n; ++i) blocks += xq_cdiv(tiles[i], (int64_t)kStreamWaves * rt) * splits[i];
        const double c = stream_run_us(blocks, rt, steps, mt);
        if (cost == 0 || c < cost) { cost = c; best = rt; }
    }
    if (us) *us = cost;
    return best;
}
// steps of a split at most (128 KB of x slice)
static int stream_steps_max(int64_t M) { return M <= 16 ? 32 : M <= 32 ? 16 : 8; }
// K splits of a forward, by its own shape: the cheapest sum of that and of the partial sums' trip (written and read back, ~6
// TB/s)
static int make_stream_splits(int64_t M, int64_t N, int64_t K) {
    const int ct = (int)(K >> 7), tiles = (int)(N / 16);
    const int mt = M <= 16 ? 1 : M <= 32 ? 2 : 4;
    int best = 0, last_steps = 0;
    double best_cost = 0;
    // (a contraction so long that its x slices need more than 64 splits takes the fewest that hold them)
    for (int s = (int)xq_cdiv(ct, stream_steps_max(M)); s <= ct && (s <= 64 || best == 0); ++s) {
        const int steps = (int)xq_cdiv(ct, s);
        if (steps == last_steps) continue;                         // more splits, none of them shorter
        last_steps = steps;
        double c;
        stream_row_tiles(&tiles, &s, 1, steps, mt, 3, &c);
        c += (double)s * M * N * 8.0 / 6.0e6;
        if (best == 0 || c < best_cost) { best = s; best_cost = c; }
    }
    return best;
}

static int stream_splits(int64_t M, int64_t N, int64_t K) {
    static thread_local PlanSlot<int> kept[64];
    const PlanKey key{M, N, K, num_cus(), 0};
    PlanSlot<int>& e = kept[key.slot()];
    if (!(e.key == key)) e = PlanSlot<int>{key, make_stream_splits(M, N, K)};
    return e.value;
}

// whether a forward of this shape runs on the two launches of this file (and not in one, xq_skinny_rows.hip)
bool skinny_takes_stream(const xq_weight* w, int64_t M, const void* lora_A, const void* lora_B, int lora_dtype, int r) {
    return skinny_supported(w, M) && !(skinny_rows_enabled() && skinny_rows_supported(w, M, lora_A, lora_B, lora_dtype, r));
}

int64_t skinny_workspace_bytes(int64_t M, int64_t N, int64_t K, int r_pad) {
    if (K < 128 || N < 16) return 256;
    const int rp = r_pad ? r_pad : 16;
    const int s = stream_splits(M, N, K);
    return al256((int64_t)s * M * N * 4) + al256((K >> 7) * M * rp * 4) + 256;
}

bool skinny_supported(const xq_weight* w, int64_t M) {
    if (M < 1 || M > 64 || w->num_experts != 1) return false;
    if (w->format == XQ_FMT_NF4 && (w->group != 64 || w->scale_dtype != XQ_SCALE_F32)) return false;   // other nf4 storages take the tile kernels
    if (w->format != XQ_FMT_FP8 && w->layout != XQ_LAYOUT_FLAT) return false;
    if (w->cols % 128 != 0 || w->cols < 1024 || w->rows % 16 != 0) return false;
    if (w->format == XQ_FMT_INT4 && (w->group % 8 != 0)) return false;
    return true;
}

// (the storages that xq_validate_weight and skinny_supported leave: nf4 fp32, nvfp4 e4m3 or fp32, int4 fp32 or bf16)
static int scale_mode(const xq_weight* w) {
    if (w->format == XQ_FMT_FP8) return kScFp8;
    if (w->format == XQ_FMT_NF4) return kScDealt;
    if (w->format == XQ_FMT_NVFP4) return w->scale_dtype == XQ_SCALE_E4M3 ? kScDealt : kScStep;
    if (w->group == 128 && w->scale_dtype == XQ_SCALE_BF16) return kScInt4Window;
    return w->group % 32 == 0 && w->cols % w->group == 0 ? kScStep : kScUse;
}

// (the uncommon scale storages keep more registers per row tile)
template <int SC>
constexpr int kRowTilesMax = SC == kScUse ? 1 : SC == kScStep ? 2 : 3;

template <int FMT, int SC, int MT, int RT>
static int launch_stream_one(const StreamBatch& b, const int* first, const bf16_t* x, int64_t ldx, int64_t M, int64_t K, size_t lds, hipStream_t s) {
    static std::atomic<bool> attr_set{false};
    if (!attr_set) {
        const hipError_t e = hipFuncSetAttribute((const void*)stream_split_kernel<FMT, SC, MT, RT>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) {
            xq_set_error("xq_linear_fwd: cannot raise the dynamic LDS limit: %s", hipGetErrorString(e));
            return XQ_ERR_LAUNCH;
        }
        attr_set = true;
    }
    stream_split_kernel<FMT, SC, MT, RT><<<(unsigned)first[4], 64 * kStreamWaves, lds, s>>>(x, (int32_t)ldx, (int32_t)M, (int32_t)K, first[1], first[2], first[3], b);
    return XQ_OK;
}
template <int FMT, int SC, int MT>
static int launch_stream_mt(const StreamBatch& b, const int* first, const bf16_t* x, int64_t ldx, int64_t M, int64_t K, int rt, size_t lds, hipStream_t s) {
    constexpr int most = kRowTilesMax<SC>;
    if constexpr (most > 2)
        if (rt == 3) return launch_stream_one<FMT, SC, MT, 3>(b, first, x, ldx, M, K, lds, s);
    if constexpr (most > 1)
        if (rt == 2) return launch_stream_one<FMT, SC, MT, 2>(b, first, x, ldx, M, K, lds, s);
    return launch_stream_one<FMT, SC, MT, 1>(b, first, x, ldx, M, K, lds, s);
}
template <int FMT, int SC>
static int launch_stream_sc(const StreamBatch& b, const int* first, const bf16_t* x, int64_t ldx, int64_t M, int64_t K, int rt, size_t lds, hipStream_t s) {
    if (M <= 16) return launch_stream_mt<FMT, SC, 1>(b, first, x, ldx, M, K, rt, lds, s);
    if (M <= 32) return launch_stream_mt<FMT, SC, 2>(b, first, x, ldx, M, K, rt, lds, s);
    return launch_stream_mt<FMT, SC, 4>(b, first, x, ldx, M, K, rt, lds, s);
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
    const int sc = scale_mode(w0), mt = M <= 16 ? 1 : M <= 32 ? 2 : 4;
    XQ_REQUIRE(ldx < (1ll << 31), "xq_linear_fwd: internal error: shape not supported by the streaming kernel");
    StreamBatch b{};
    EpiBatch e{};
    uint8_t* ws = (uint8_t*)workspace;
    bool vec = true;
    int steps = 0;
    for (int i = 0; i < n_jobs; ++i) {
        const SkinnyRowsJob& j = jobs[i];
        const int rp = j.r > 0 ? (j.r + 15) / 16 * 16 : 0;
        const int64_t N = j.w->rows;
        StreamJob& g = b.job[i];
        g.splits = stream_splits(M, N, K);
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
    const int rt = stream_row_tiles(tiles, splits, n_jobs, steps, mt, sc == kScUse ? kRowTilesMax<kScUse> : sc == kScStep ? kRowTilesMax<kScStep> : 3, nullptr);
    int first[5] = {0, 0, 0, 0, 0}, efirst[5] = {0, 0, 0, 0, 0};
    for (int i = 0; i < kStreamJobs; ++i) {
        first[i + 1] = first[i];
        efirst[i + 1] = efirst[i];
        if (i < n_jobs) {
            b.job[i].row_blocks = (int)xq_cdiv(tiles[i], (int64_t)kStreamWaves * rt);
            first[i + 1] += b.job[i].row_blocks * b.job[i].splits;
            efirst[i + 1] += (int)xq_cdiv(b.job[i].N, 128);
        } else {
            b.job[i] = b.job[0];
            e.job[i] = e.job[0];
        }
    }
    const size_t lds = (size_t)steps * mt * 4096 + 64;             // the x slice of the longest split, the nf4 levels
    int rc = XQ_ERR_UNSUPPORTED;
#define XQ_STREAM_CASE(F, S) \
    if (w0->format == F && sc == S) rc = launch_stream_sc<F, S>(b, first, x, ldx, M, K, rt, lds, stream)
    XQ_STREAM_CASE(XQ_FMT_FP8, kScFp8);
    XQ_STREAM_CASE(XQ_FMT_INT4, kScInt4Window);
    XQ_STREAM_CASE(XQ_FMT_INT4, kScStep);
    XQ_STREAM_CASE(XQ_FMT_INT4, kScUse);
    XQ_STREAM_CASE(XQ_FMT_NVFP4, kScDealt);
    XQ_STREAM_CASE(XQ_FMT_NVFP4, kScStep);
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
    const unsigned threads = M < 4 && rw == 1 ? (unsigned)M * 64 : 256;
    const dim3 grid(cols, (unsigned)xq_cdiv(M, 4 * rw));
#define XQ_EPI(RW)                                                                                                                             \
    do {                                                                                                                                       \
        if (swiglu) {                                                                                                                          \
            if (vec) stream_epilogue_kernel<RW, true, true><<<grid, threads, 0, stream>>>((int)M, efirst[1], efirst[2], efirst[3], e);         \
            else stream_epilogue_kernel<RW, false, true><<<grid, threads, 0, stream>>>((int)M, efirst[1], efirst[2], efirst[3], e);            \
        } else {                                                                                                                               \
            if (vec) stream_epilogue_kernel<RW, true, false><<<grid, threads, 0, stream>>>((int)M, efirst[1], efirst[2], efirst[3], e);        \
            else stream_epilogue_kernel<RW, false, false><<<grid, threads, 0, stream>>>((int)M, efirst[1], efirst[2], efirst[3], e);           \
        }                                                                                                                                      \
    } while (0)
    if (rw == 1) XQ_EPI(1);
    else if (rw == 2) XQ_EPI(2);
    else XQ_EPI(4);
#undef XQ_EPI
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
    // M <= 16: one launch, whole rows per block, where the shape and the LoRA operands fit it and a slot is free
    int rc = XQ_ERR_UNSUPPORTED;
    if (g_skinny_rows && skinny_rows_supported(w, M, lora_A, lora_B, lora_dtype, r))
        rc = launch_skinny_rows(w, x, ldx, M, lora_A, lora_B, r, scaling, bias, y, ldy, workspace, stream);
    if (rc == XQ_ERR_UNSUPPORTED) {
        const SkinnyRowsJob job{w, lora_A, lora_B, rp ? r : 0, scaling, bias, y, ldy};
        rc = launch_skinny_stream(&job, 1, false, x, ldx, M, lora_dtype, workspace, stream);
    }
    if (timed) xq_profile_mark_end(stream);
    if (rc) return rc;
    XQ_CHECK_LAUNCH("skinny forward");
    return XQ_OK;
}

}  // namespace xq
