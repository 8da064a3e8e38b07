// Fused dequant-GEMM for dense weights from 65 rows on, wherever it is the shorter one by the estimates (xq_gemm.hip: most products of
// some hundreds of rows, narrow ones of thousands): every weight value is decoded by exactly one wave per 32 MW rows, in registers,
// straight into the operand of v_mfma_f32_32x32x16_bf16.
//
//   C[rows, Nout] = A[rows, Kc] . Wop (+ su[rows, r] . right[Nout, r]^T) (+ bias)
//     CC  (forward): Wop[kc][n] = W[n][kc]        !CC (dgrad): Wop[kc][n] = W[kc][n]
//
//  * A block owns 32 MW rows x 256 columns: four waves side by side, 64 columns each, twice: the two halves of the waves take the
//    two halves (phases) of the block's share of the contraction, and their fp32 sums meet in LDS at the end.  A wave's tile is
//    MW x 2 MFMA tiles (128 accumulator registers at MW = 4).
//  * Per 16 of the contraction a wave decodes two weight operands (~21 vector instructions each) for 2 MW MFMAs of 32 cycles.
//    Why 32 x 32 x 16: an MFMA takes two issue slots of the vector unit in either form, and this one lasts twice as long: 8 of them
//    hide 48 vector instructions of the SIMD's two waves (274 cycles for 256 of matrix work), 16 of the 16 x 16 x 32 form only 32
//    (48: 378 cycles).
//  * Activations: direct-to-LDS loads of [32 MW rows][64 k] per phase, two stages; 16-byte chunk c of row r at chunk
//    c ^ ((r >> 1) & 7).
//  * Weights come as their codes by direct-to-LDS loads too.  CC: [256 n][64 bytes], one 16-byte piece of its row per lane and read
//    (4-bit: 64 bytes are two steps' codes and are loaded every other step).  Loaded into registers instead (16 rows x 64 bytes or
//    32 rows x 32 bytes a load) the same bytes held the step at 2.2 us where it now takes 1.25 (64 tiles, block-fp8).
//    !CC: [64 kc][256 n] as in memory; the transposing byte read ds_read_b64_tr_b8 hands a lane eight rows of one byte column: one
//    operand of block-fp8, or the operands of the two columns that share a 4-bit byte (so a wave's two tiles hold its even and odd
//    columns); scales, one per row and column group, pass through LDS as [group][row], int4 ones as 512 s and -8 s.
//  * One barrier per half step of 32 k: phase 1 runs half a step behind phase 0, so that one phase's LDS latency and first decode at
//    a step boundary lie under the other's MFMAs (forward, 64 tiles: 1.33 -> 1.19 us a step without the loads).  A step's loads are
//    requested at the start of the step before it and waited for at its end.
//  * What bounds it: with every compute unit at work the step of 128 x 256 x 2 x 64 takes 1.55-1.65 us, 1.3 PFLOP/s, the rate that
//    power leaves the MFMA; around the steps lie 8-10 us (launch 2.5, first loads 1-3, the phases' meeting 2, the output 1.4-2.5)
//    and, where the contraction is split over blocks, the trip of the fp32 sums.  nf4 is bound by its level look-ups (one LDS read
//    a weight: 2.2-2.5 us a step).
//    int4 [4096, 4096], 512 rows: 42.6 -> 35.0 us forward, 39.3 -> 34.3 dgrad; [12288, 4096] 93.8 -> 56.8, 82.5 -> 64.1 (against 128
//    x 128 tiles decoded into LDS on the 32 x 32 x 16 form by each of the row tiles); more at plan_mid (xq_gemm.hip).
#pragma once

#include "xq_gemm_dtl.h"
#include "xq_skinny.h"

namespace xq {

template <int FMT, bool CC, int MW>
struct GeoMid {
    static constexpr int NT = 512, BM = 32 * MW, BN = 256, KP = 2;
    static constexpr int BK = 64;                                                          // contraction of a step
    static constexpr int WS = CC && FMT != XQ_FMT_FP8 ? 2 : 1;                             // steps whose codes come together: 64 bytes of a row
    static constexpr int XC = BK / 8;                                                      // 16-byte chunks of an activation row
    static constexpr int X_BYTES = BM * BK * 2;                                            // of a phase and stage
    static constexpr int W_PITCH = CC ? 64 : FMT == XQ_FMT_FP8 ? BN : BN / 2;              // bytes of a row of codes in LDS
    static constexpr int W_BYTES = (CC ? BN : BK) * W_PITCH;
    static constexpr int S_BYTES = CC || FMT == XQ_FMT_FP8 ? 0 : FMT == XQ_FMT_NF4 ? 4 * BK * 4 : FMT == XQ_FMT_INT4 ? 2 * 2 * BK * 4 : 16 * BK;
    static constexpr int PHASE_BYTES = X_BYTES + W_BYTES + S_BYTES, STAGE_BYTES = KP * PHASE_BYTES;
    static constexpr int RED_PITCH = BN + 4;
    static constexpr int SCL_MAX = 256;                                                    // block-fp8: 128-k blocks of the contraction
    static constexpr int HEAD = FMT == XQ_FMT_NF4 ? 256 : 0;                               // the nf4 levels, where a look-up needs no address of its own
    static constexpr size_t loop_bytes() { return HEAD + 2 * (size_t)STAGE_BYTES + (FMT == XQ_FMT_FP8 ? 2 * SCL_MAX * 4 : 0); }
    static constexpr size_t lds_bytes() { return loop_bytes() > (size_t)BM * RED_PITCH * 4 ? loop_bytes() : (size_t)BM * RED_PITCH * 4; }
};

typedef uint32_t mid_u32_a1 __attribute__((aligned(1)));
typedef u32x2 u32x2_a1 __attribute__((aligned(1)));

template <int FMT, bool CC, int MW>
__global__ void __launch_bounds__(512, 2) gemm_mid_kernel(G256Args g) {
    using D = GeoMid<FMT, CC, MW>;
    constexpr int EB = FMT == XQ_FMT_FP8 ? 1 : 2;                     // codes per byte
    extern __shared__ __attribute__((aligned(16))) unsigned char msm[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ph = wave >> 2, wn = wave & 3;                          // phase, column group
    const int l32 = lane & 31, h = lane >> 5;

    int pid_m, pid_n;
    {
        // an XCD takes a contiguous range of the tiles, the row tiles of a column tile next to each other
        const int nb = g.tiles_m * g.tiles_n;
        const int b = blockIdx.x, per = nb >> 3;
        const int logical = (b < per * 8) ? (b & 7) * per + (b >> 3) : b;
        pid_n = logical / g.tiles_m;
        pid_m = logical - pid_n * g.tiles_m;
    }
    const int64_t row0 = (int64_t)pid_m * D::BM;
    const int n0 = pid_n * D::BN;
    const int split = blockIdx.y;
    // this phase's K-steps: the contraction in 2 ksplit ranges, the first `rem` of them one step longer
    const int nk_all = g.Kc / D::BK, units = nk_all / D::WS, parts = g.ksplit * D::KP, q_units = units / parts, rem = units - q_units * parts;
    const int v = split * D::KP + ph;
    const int kt0 = (v * q_units + min(v, rem)) * D::WS, nk = (q_units + (v < rem ? 1 : 0)) * D::WS;
    const int n_loop = (q_units + (split * D::KP < rem ? 1 : 0)) * D::WS;

    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)msm;
    const auto phase_at = [&](int stage) { return (uint32_t)(D::HEAD + stage * D::STAGE_BYTES + ph * D::PHASE_BYTES); };

    // ---- direct-to-LDS sources of this wave: its activation rows, !CC: its share of the K-step's codes
    constexpr int XL = D::X_BYTES / 4096, XC = D::XC, XR = 64 / XC;                   // loads of a wave, chunks of a row, rows of a load
    const auto x_sw = [](int r) { return (r >> 1) & 7; };
    uint32_t a_off[XL];
#pragma unroll
    for (int i = 0; i < XL; ++i) {
        const int r = (wn * XL + i) * XR + lane / XC;
        const int64_t row = min(row0 + r, g.M - 1);
        a_off[i] = (uint32_t)((row * g.lda + (((lane % XC) ^ x_sw(r)) << 3)) * 2);
    }
    constexpr int WL = D::W_BYTES / 4096, CPR = D::W_PITCH / 16;             // loads of a wave, 16-byte chunks of a row
    uint32_t w_off[WL > 0 ? WL : 1];
    if constexpr (CC) {
#pragma unroll
        for (int i = 0; i < WL; ++i) {
            const int r = (wn * WL + i) * 16 + (lane >> 2);
            w_off[i] = (uint32_t)((int64_t)min(n0 + r, g.wrows - 1) * (g.wcols / EB) + (((lane & 3) ^ ((r >> 2) & 3)) << 4));
        }
    } else {
#pragma unroll
        for (int i = 0; i < WL; ++i) {
            const int r = (wn * WL + i) * (64 / CPR) + lane / CPR, c = lane % CPR;
            const int sw = CPR == 16 ? (r & 7) << 1 : ((r >> 1) & 3) << 1;
            const int col = min(n0 / EB + ((c ^ sw) << 4), g.wcols / EB - 16);
            w_off[i] = (uint32_t)((int64_t)r * (g.wcols / EB) + col);
        }
    }
    const int nk1 = (!CC && g.W2 != nullptr) ? g.nk1 : (1 << 30);                     // K-steps from nk1 on read the second matrix
    const auto issue = [&](int s, int stage) {
        const int kt = kt0 + min(s, nk - 1);
        const uint32_t dst = lds0 + phase_at(stage);
#pragma unroll
        for (int i = 0; i < XL; ++i)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                         :: "s"(__builtin_amdgcn_readfirstlane(dst + (wn * XL + i) * 1024)), "v"(a_off[i]), "s"(g.A + kt * D::BK) : "memory");
        if (D::WS == 1 || (s & 1) == 0) {
            // (past the phase's end: its last codes again)
            const uint8_t* base = CC ? g.W + (kt0 + min(s, nk - D::WS)) * (D::BK / EB)
                                     : kt >= nk1 ? g.W2 + (int64_t)(kt - nk1) * D::BK * (g.wcols / EB) : g.W + (int64_t)kt * D::BK * (g.wcols / EB);
            const uint32_t wdst = D::WS == 1 ? dst : lds0 + phase_at((s >> 1) & 1);
#pragma unroll
            for (int i = 0; i < WL; ++i)
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                             :: "s"(__builtin_amdgcn_readfirstlane(wdst + D::X_BYTES + (wn * WL + i) * 1024)), "v"(w_off[i]), "s"(base) : "memory");
        }
    };

    // ---- scales.  CC: of the lane's rows in tiles 0 and 1, for the two steps whose codes come together (loaded ahead, then moved to
    // the current ones); !CC: one load a thread, on its way to LDS
    uint32_t cur[2] = {}, next[2][2] = {};
    const float gs = FMT == XQ_FMT_NVFP4 ? g.global_scale[0] : 1.0f;
    uint32_t srow[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) srow[t] = (uint32_t)min(n0 + wn * 64 + t * 32 + l32, g.wrows - 1);
    const int pt = tid & 255;                                          // thread of the phase
    const auto load_s = [&](int s) {
        const int kt = kt0 + min(s, nk - 1);
        if constexpr (CC && FMT != XQ_FMT_FP8) {
            if ((s & 1) == 0) {
                const int u = kt >> 1;
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    if constexpr (FMT == XQ_FMT_INT4) next[t][0] = ((const uint16_t*)g.scales)[(int64_t)srow[t] * (g.wcols >> 7) + u];
                    else {
                        const u32x2_a1 v = *(const u32x2_a1*)(g.scales + ((int64_t)srow[t] * (g.wcols >> 7) + u) * 8);
                        next[t][0] = v[0];
                        next[t][1] = v[1];
                    }
                }
            }
        } else if constexpr (!CC) {
            const int64_t r0 = (int64_t)kt * D::BK;
            if constexpr (FMT == XQ_FMT_INT4) {                        // threads 0 .. 127: row pt & 63, group pt >> 6 of the tile's two
                const int grp = min((n0 >> 7) + ((pt >> 6) & 1), (g.wcols >> 7) - 1);
                next[0][0] = ((const uint16_t*)g.scales)[(r0 + (pt & 63)) * (g.wcols >> 7) + grp];
            } else if constexpr (FMT == XQ_FMT_NF4) {                  // row pt >> 2, group pt & 3 of four
                const int grp = min((n0 >> 6) + (pt & 3), (g.wcols >> 6) - 1);
                next[0][0] = ((const uint32_t*)g.scales)[(r0 + (pt >> 2)) * (g.wcols >> 6) + grp];
            } else if constexpr (FMT == XQ_FMT_NVFP4) {                // row pt >> 2, groups 4 (pt & 3) .. of sixteen
                const int grp = min((n0 >> 4) + (pt & 3) * 4, (g.wcols >> 4) - 4);
                next[0][0] = *(const mid_u32_a1*)(g.scales + (r0 + (pt >> 2)) * (g.wcols >> 4) + grp);
            }
        }
    };
    // !CC: the scales of a K-step into its stage
    const auto store_s = [&](int stage) {
        unsigned char* dst = msm + phase_at(stage) + D::X_BYTES + D::W_BYTES;
        if constexpr (!CC && FMT == XQ_FMT_INT4) {                     // [512 s | -8 s][group][row]
            if (pt < 128) {
                const float s = __uint_as_float(next[0][0] << 16);
                ((float*)dst)[pt] = s * 512.0f;
                ((float*)dst)[128 + pt] = s * -8.0f;
            }
        } else if constexpr (!CC && FMT == XQ_FMT_NF4) {
            ((uint32_t*)dst)[(pt & 3) * 64 + (pt >> 2)] = next[0][0];
        } else if constexpr (!CC && FMT == XQ_FMT_NVFP4) {
#pragma unroll
            for (int i = 0; i < 4; ++i) dst[((pt & 3) * 4 + i) * 64 + (pt >> 2)] = (uint8_t)(next[0][0] >> (8 * i));
        }
    };
    const float* levels = (const float*)msm;
    float* s_lds = (float*)(msm + 2 * D::STAGE_BYTES);
    if constexpr (FMT == XQ_FMT_FP8) {
        const int scols = (g.wcols + 127) >> 7, nkb = (nk_all + 1) >> 1;
        for (int i = tid; i < 2 * nkb; i += D::NT) {
            const int blk = i / nkb, kb = i - blk * nkb, nn = n0 + blk * 128;
            const bool second = 2 * kb >= nk1;                         // (nk1 is even)
            const float* sp = (const float*)(second ? g.scales2 : g.scales);
            const int kb1 = second ? kb - (nk1 >> 1) : kb;
            s_lds[blk * D::SCL_MAX + kb] = CC ? sp[(min(nn, g.wrows - 1) >> 7) * scols + kb1] : sp[(int64_t)kb1 * scols + (min(nn, g.wcols - 1) >> 7)];
        }
    } else if constexpr (FMT == XQ_FMT_NF4) {
        if (tid < 16) ((float*)msm)[tid] = kNf4Level[tid];
    }

    f32x16 acc[2][MW];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < MW; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[t][i][e] = 0.0f;

    // byte address (stage 0) of this lane's activation chunk j in row tile 0; + i * 64 BK
    constexpr int NJ = D::BK / 16;
    uint32_t xo[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int c = CC ? 4 * h + j : 2 * j + h;
        xo[j] = (uint32_t)(l32 * (D::BK * 2) + ((c ^ x_sw(l32)) << 4));
    }
    // !CC: this lane's 8-byte piece of the codes for tile t (4-bit: both tiles) and the first rows of a half step; + j * 16 rows
    typedef __attribute__((ext_vector_type(2))) int i32x2;
    const int sub = (lane >> 4) & 1, l16 = lane & 15, rw = 8 * h + (l16 >> 1);
    const auto tr_read = [&](const unsigned char* base, int t, int j) {
        const int r = 16 * j + rw, sw = CPR == 16 ? (r & 7) << 1 : ((r >> 1) & 3) << 1;
        const int c = (FMT == XQ_FMT_FP8 ? wn * 4 + t * 2 : wn * 2) + sub;
        const unsigned char* p = base + r * D::W_PITCH + ((c ^ sw) << 4) + ((l16 & 1) << 3);
        const i32x2 x = __builtin_amdgcn_ds_read_tr8_b64_v2i32((i32x2 __attribute__((address_space(3)))*)p);
        return u32x2{(uint32_t)x[0], (uint32_t)x[1]};
    };

    bf16x8 xf[2][MW], wf[2][2];
    u32x2 raw[!CC && FMT == XQ_FMT_NF4 ? 4 : 2][2];
    u32x4 raw8[2][2];
    float lv[2][FMT == XQ_FMT_NF4 ? 16 : 1];                           // nf4: the levels of a half step's codes
    f32x4 fsc[2][4];
    // half of a step: 32 k; operands are decoded and read one 16-k piece ahead of their MFMAs
    const auto half_step = [&](int s, int stage, auto HALF_) {
        constexpr int HALF = decltype(HALF_)::value;
        const unsigned char* xs = msm + phase_at(stage);
        float fs = 1.0f;
        if constexpr (FMT == XQ_FMT_FP8) fs = s_lds[(wn >> 1) * D::SCL_MAX + ((kt0 + s) >> 1)];
        const auto load_xf = [&](int j, int b) {
#pragma unroll
            for (int i = 0; i < MW; ++i) xf[b][i] = *(const bf16x8*)(xs + xo[j] + i * (64 * D::BK));
        };
        // what the decode of half step j reads from LDS, requested one half step before it
        const auto fetch = [&](int j) {
            if constexpr (CC) {                                        // a 16-byte piece of the lane's row: two half steps (4-bit: four)
                constexpr int JP = FMT == XQ_FMT_FP8 ? 2 : 4;
                if (j % JP == 0) {
                    const int c = FMT == XQ_FMT_FP8 ? 2 * h + j / JP : 2 * stage + h;      // (4-bit: the step's parity is its stage)
                    const unsigned char* ws = msm + phase_at(D::WS == 1 ? stage : (s >> 1) & 1) + D::X_BYTES;
#pragma unroll
                    for (int t = 0; t < 2; ++t)
                        raw8[j / JP][t] = *(const u32x4*)(ws + (wn * 64 + t * 32 + l32) * 64 + ((c ^ ((l32 >> 2) & 3)) << 4));
                }
                if constexpr (FMT == XQ_FMT_NF4) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) lv[j & 1][i] = levels[(raw8[0][i >> 3][j] >> (4 * (i & 7))) & 0xfu];
                }
            } else if constexpr (!CC && FMT == XQ_FMT_FP8) {
#pragma unroll
                for (int t = 0; t < 2; ++t) raw[j & 1][t] = tr_read(xs + D::X_BYTES, t, j);
            } else if constexpr (!CC) {
                if constexpr (FMT == XQ_FMT_NF4) {
                    if (j == 0) {
#pragma unroll
                        for (int k = 0; k < 4; ++k) raw[k][0] = tr_read(xs + D::X_BYTES, 0, k);
                    }
#pragma unroll
                    for (int i = 0; i < 16; ++i) lv[j & 1][i] = levels[(raw[j][0][(i >> 2) & 1] >> (8 * (i & 3) + 4 * (i >> 3))) & 0xfu];
                } else {
                    raw[j & 1][0] = tr_read(xs + D::X_BYTES, 0, j);
                }
                const unsigned char* sp = xs + D::X_BYTES + D::W_BYTES;
                if constexpr (FMT == XQ_FMT_NVFP4) {
                    raw[j & 1][1] = *(const u32x2*)(sp + (wn * 4 + (l32 >> 3)) * 64 + 16 * j + 8 * h);
                } else {
                    const float* f = (const float*)sp + (FMT == XQ_FMT_INT4 ? wn >> 1 : wn) * 64 + 16 * j + 8 * h;
                    fsc[j & 1][0] = *(const f32x4*)f;
                    fsc[j & 1][1] = *(const f32x4*)(f + 4);
                    if constexpr (FMT == XQ_FMT_INT4) {
                        fsc[j & 1][2] = *(const f32x4*)(f + 128);
                        fsc[j & 1][3] = *(const f32x4*)(f + 132);
                    }
                }
            }
        };
        const auto decode = [&](int j, int b) {
            if constexpr (CC) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    if constexpr (FMT == XQ_FMT_FP8) {
                        wf[b][t] = decode8<FMT>(raw8[j >> 1][t][2 * (j & 1)], raw8[j >> 1][t][2 * (j & 1) + 1], fs, 0.0f);
                    } else {
                        const uint32_t w = raw8[0][t][j];
                        if constexpr (FMT == XQ_FMT_INT4) {
                            const float sc = __uint_as_float(cur[t] << 16);
                            wf[b][t] = decode8<FMT>(w, 0u, sc, -8.0f * sc);
                        } else if constexpr (FMT == XQ_FMT_NVFP4) {
                            wf[b][t] = decode8<FMT>(w, 0u, e4m3_to_f32((uint8_t)(cur[t] >> (8 * (j >> 1)))) * gs, 0.0f);
                        } else {
                            const float sc = __uint_as_float(cur[t]);
                            const float* l = lv[j & 1] + 8 * t;
                            wf[b][t] = __builtin_bit_cast(bf16x8, u32x4{pack_bf16x2(l[0] * sc, l[1] * sc), pack_bf16x2(l[2] * sc, l[3] * sc),
                                                                        pack_bf16x2(l[4] * sc, l[5] * sc), pack_bf16x2(l[6] * sc, l[7] * sc)});
                        }
                    }
                }
            } else if constexpr (FMT == XQ_FMT_FP8) {
#pragma unroll
                for (int t = 0; t < 2; ++t) wf[b][t] = decode8<FMT>(raw[j & 1][t][0], raw[j & 1][t][1], fs, 0.0f);
            } else {
                const u32x2 w = raw[FMT == XQ_FMT_NF4 ? j : j & 1][0];
                float e[8], o[8];                                      // the lane's even and odd column, eight rows
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    if constexpr (FMT == XQ_FMT_INT4) {
                        const f32x4 a = fsc[j & 1][u], c = fsc[j & 1][2 + u];
                        const uint32_t ev = w[u] & 0x0f0f0f0fu, od = (w[u] >> 4) & 0x0f0f0f0fu;
                        const f32x2 e01 = e4m3x2_to_f32(ev, false), e23 = e4m3x2_to_f32(ev, true);
                        const f32x2 o01 = e4m3x2_to_f32(od, false), o23 = e4m3x2_to_f32(od, true);
                        e[4 * u] = __builtin_fmaf(e01[0], a[0], c[0]); e[4 * u + 1] = __builtin_fmaf(e01[1], a[1], c[1]);
                        e[4 * u + 2] = __builtin_fmaf(e23[0], a[2], c[2]); e[4 * u + 3] = __builtin_fmaf(e23[1], a[3], c[3]);
                        o[4 * u] = __builtin_fmaf(o01[0], a[0], c[0]); o[4 * u + 1] = __builtin_fmaf(o01[1], a[1], c[1]);
                        o[4 * u + 2] = __builtin_fmaf(o23[0], a[2], c[2]); o[4 * u + 3] = __builtin_fmaf(o23[1], a[3], c[3]);
                    } else if constexpr (FMT == XQ_FMT_NVFP4) {
                        const u32x2 sb = raw[j & 1][1];
                        const f32x2 s01 = e4m3x2_to_f32(sb[u], false), s23 = e4m3x2_to_f32(sb[u], true);
                        const f32x2 x0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w[u], 1.0f, 0), x1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w[u], 1.0f, 1);
                        const f32x2 x2 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w[u], 1.0f, 2), x3 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w[u], 1.0f, 3);
                        const float s0 = s01[0] * gs, s1 = s01[1] * gs, s2 = s23[0] * gs, s3 = s23[1] * gs;
                        e[4 * u] = x0[0] * s0; e[4 * u + 1] = x1[0] * s1; e[4 * u + 2] = x2[0] * s2; e[4 * u + 3] = x3[0] * s3;
                        o[4 * u] = x0[1] * s0; o[4 * u + 1] = x1[1] * s1; o[4 * u + 2] = x2[1] * s2; o[4 * u + 3] = x3[1] * s3;
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            e[4 * u + i] = lv[j & 1][4 * u + i] * fsc[j & 1][u][i];
                            o[4 * u + i] = lv[j & 1][8 + 4 * u + i] * fsc[j & 1][u][i];
                        }
                    }
                }
                wf[b][0] = __builtin_bit_cast(bf16x8, u32x4{pack_bf16x2(e[0], e[1]), pack_bf16x2(e[2], e[3]), pack_bf16x2(e[4], e[5]), pack_bf16x2(e[6], e[7])});
                wf[b][1] = __builtin_bit_cast(bf16x8, u32x4{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]), pack_bf16x2(o[4], o[5]), pack_bf16x2(o[6], o[7])});
            }
        };
        if constexpr (HALF == 0) {
            fetch(0);
            load_xf(0, 0);
            fetch(1);
            decode(0, 0);
        }
#pragma unroll
        for (int j = HALF * (NJ / 2); j < (HALF + 1) * (NJ / 2); ++j) {
            __builtin_amdgcn_sched_barrier(0);
            if (j + 1 < NJ) {
                load_xf(j + 1, (j + 1) & 1);
                decode(j + 1, (j + 1) & 1);
            }
            if (j + 2 < NJ) fetch(j + 2);
#pragma unroll
            for (int i = 0; i < MW; ++i)
#pragma unroll
                for (int t = 0; t < 2; ++t) acc[t][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[j & 1][t], xf[j & 1][i], acc[t][i], 0, 0, 0);
            // between the MFMAs: the next operands' reads, then their decode
#pragma unroll
            for (int i = 0; i < 2 * MW; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
            }
        }
    };
    // the scales of step s become the current ones, waited for here, where only one step's loads are out (CC), or go to LDS (!CC)
    const auto take_s = [&](int s, int stage) {
        if constexpr (CC && FMT != XQ_FMT_FP8) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const uint32_t d = FMT == XQ_FMT_INT4 ? next[t][0] : next[t][stage];
                cur[t] = FMT == XQ_FMT_NVFP4 ? d >> (16 * h) : d;
                asm volatile("" : "+v"(cur[t]));
            }
        } else if constexpr (!CC) {
            store_s(stage);
        }
    };

    issue(0, 0);
    load_s(0);
    take_s(0, 0);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    using H0 = std::integral_constant<int, 0>;
    using H1 = std::integral_constant<int, 1>;
    // Phase 1 runs half a step behind: where one phase crosses a step boundary (its fragments' LDS latency and first decode
    // exposed) the other one is in the middle of its MFMAs.
    const auto first_half = [&](int s, int par) {
        if (s + 1 < n_loop) {
            load_s(s + 1);
            issue(s + 1, par ^ 1);
        }
        if (s < nk) half_step(s, par, H0{});
    };
    const auto second_half = [&](int s, int par) {
        if (s < nk) half_step(s, par, H1{});
        if (s + 1 < n_loop) take_s(s + 1, par ^ 1);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    };
    const auto meet = [&]() { asm volatile("s_barrier" ::: "memory"); };
    if (ph == 1) meet();
    int s = 0;
#pragma unroll 1
    for (; s + 2 <= n_loop; s += 2) {
        first_half(s, 0); meet();
        second_half(s, 0); meet();
        first_half(s + 1, 1); meet();
        second_half(s + 1, 1); meet();
    }
    if (s < n_loop) {
        first_half(s, 0); meet();
        second_half(s, 0); meet();
    }
    if (ph == 0) meet();

    // ---- low-rank side term: the 16-rank steps dealt to the phases
    if (g.r_pad > 0 && split == 0) {
#pragma unroll 1
        for (int ks = ph; ks < (g.r_pad >> 4); ks += D::KP) {
            bf16x8 wl[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int nl = CC || FMT == XQ_FMT_FP8 ? t * 32 + l32 : 2 * l32 + t;
                wl[t] = __builtin_bit_cast(bf16x8, right_chunk(g.right, -1, min(n0 + wn * 64 + nl, g.Nout - 1), ks * 2 + h));
            }
#pragma unroll
            for (int i = 0; i < MW; ++i) {
                const bf16x8 xl = *(const bf16x8*)(g.su + min(row0 + i * 32 + l32, g.M - 1) * g.ld_su + ks * 16 + h * 8);
#pragma unroll
                for (int t = 0; t < 2; ++t) acc[t][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wl[t], xl, acc[t][i], 0, 0, 0);
            }
        }
    }

    // ---- the phases' sums meet: [row][column] fp32 in LDS; phase 1 leaves the first MW / 2 row tiles to phase 0 and takes the others
    float* red = (float*)msm;
    constexpr int MH = MW / 2;
    const auto at = [&](int i, int q) { return red + (i * 32 + l32) * D::RED_PITCH + wn * 64 + (CC || FMT == XQ_FMT_FP8 ? 8 * q + 4 * h : 16 * q + 8 * h); };
    const auto put = [&](int i) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if constexpr (CC || FMT == XQ_FMT_FP8) {
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    *(f32x4*)(at(i, q) + t * 32) = f32x4{acc[t][i][4 * q], acc[t][i][4 * q + 1], acc[t][i][4 * q + 2], acc[t][i][4 * q + 3]};
            } else {                                                   // the tiles hold alternate columns
                *(f32x4*)at(i, q) = f32x4{acc[0][i][4 * q], acc[1][i][4 * q], acc[0][i][4 * q + 1], acc[1][i][4 * q + 1]};
                *(f32x4*)(at(i, q) + 4) = f32x4{acc[0][i][4 * q + 2], acc[1][i][4 * q + 2], acc[0][i][4 * q + 3], acc[1][i][4 * q + 3]};
            }
        }
    };
    const auto add = [&](int i) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                if constexpr (CC || FMT == XQ_FMT_FP8) {
                    const f32x4 p = *(const f32x4*)(at(i, q) + t * 32);
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[t][i][4 * q + e] += p[e];
                } else {
                    const f32x4 p = *(const f32x4*)(at(i, q) + 4 * t);
                    acc[0][i][4 * q + 2 * t] += p[0]; acc[1][i][4 * q + 2 * t] += p[1];
                    acc[0][i][4 * q + 2 * t + 1] += p[2]; acc[1][i][4 * q + 2 * t + 1] += p[3];
                }
            }
    };
    // (the last iteration's barrier lies behind every read of the stages)
#pragma unroll
    for (int i = 0; i < MW; ++i)
        if ((i < MH) == (ph == 1)) put(i);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MW; ++i)
        if ((i < MH) != (ph == 1)) { add(i); put(i); }
    __syncthreads();

    // ---- out: whole rows of the tile, 8 columns a thread
    const int c8 = (tid & 31) * 8, n = n0 + c8;
    if (n >= g.Nout) return;                                           // (Nout % 16 == 0)
    float bias[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (g.bias && split == 0) {
#pragma unroll
        for (int e = 0; e < 8; ++e) bias[e] = bf16_to_f32(g.bias[n + e]);
    }
#pragma unroll 4
    for (int r = tid >> 5; r < D::BM; r += 16) {
        const int64_t row = row0 + r;
        if (row >= g.M) break;
        f32x4 a = *(const f32x4*)(red + r * D::RED_PITCH + c8), b = *(const f32x4*)(red + r * D::RED_PITCH + c8 + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) { a[e] += bias[e]; b[e] += bias[4 + e]; }
        if (g.ksplit > 1) {
            float* p = g.partial + ((int64_t)split * g.M + row) * g.Nout + n;
            *(f32x4*)p = a;
            *(f32x4*)(p + 4) = b;
        } else {
            bf16_t* c = g.C + row * g.ldc + n;
            const u32x4 o = {pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3]), pack_bf16x2(b[0], b[1]), pack_bf16x2(b[2], b[3])};
            if (g.wide_rows) {
                *(u32x4*)c = o;
            } else {
                *(u32x2*)c = u32x2{o[0], o[1]};
                *(u32x2*)(c + 4) = u32x2{o[2], o[3]};
            }
        }
    }
}

}  // namespace xq
