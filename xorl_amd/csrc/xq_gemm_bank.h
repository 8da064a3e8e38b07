// Fused dequant-GEMM over expert banks of block-fp8 and nvfp4 (e4m3 scales of 16 rows), and over dense block-fp8 weights: tiles of 128 routed rows x 256 columns, four waves side by side (a wave 128 x
// 64), two blocks on a compute unit.
//
//   C[rows, Nout] = A[rows, Kc] . Wop[e] (+ su[rows, r] . Lr[e][Nout, r]^T)
//     !CC (a bank's forward): Wop[kc][n] = W[e][kc][n]; optionally two banks side by side (G256Args: W2, ncols1)
//      CC (a bank's dgrad):   Wop[kc][n] = W[e][n][kc]; optionally one sum over two banks (K-steps from nk1 on read the second;
//                             nvfp4: the two products side by side)
//     DENSE (block-fp8): one weight, all rows, or two of one shape on one input; CC forward [Nout, Kc], !CC dgrad; the right-hand factor as it
//                             is, and a bias
//
// Decode and order of sums are gemm_dtl16_kernel's for block-fp8 (xq_gemm_dtl.h), and so are the fragments: one 16-byte piece of a
// weight row, or two transposing byte reads, is a lane's operand of both k32 steps of a K-step.  nvfp4 bytes hold rows 2 p and 2 p + 1
// of a column.  !CC: one transposing read is a lane's 16 k of its column, under one scale.  CC: a lane's 16 bytes are its 16 k of an
// even and an odd output column, which are two tiles of a pair (a lane ends with eight columns in a row, without a swap), and both share
// 16 scales.
//
// What bounds it: the vector instructions of the decode beside the MFMAs, and the chip's power.  A wave's K-step is 64 MFMAs (1024
// cycles) and 140 vector instructions; alone on its SIMD it takes 2070 cycles, two waves side by side 2780 for both (256 x 256 tiles of one
// block: 3300), at 1.85 GHz.  Measured on the way, for the four launches of a routed MLP of 128 experts 2048/768 and 131072 rows:
// 2555 us with 256 x 256 tiles, one block a unit (12 of 30 us of a tile of 12 K-steps outside the loop: nothing overlaps them there),
// 2420 as 128 x 256 tiles, 2250 as it stands (0.83-1.07 -> 0.97-1.2 PFLOP/s).  nvfp4, forward and backward of such an MLP, against decoded
// tiles in LDS (gemm_256_kernel): 4400 -> 3680 us, 32768 rows 1581 -> 1122, 16384 rows 1032 -> 755; with gate, up and the dgrad of down left there, for
// their order of sums: 4443 -> 4034, 1547 -> 1350, 998 -> 884, and without a backward, 76800 rows 1232 -> 905.
// Dense block-fp8 MLP 4096/12288 of 2048 rows (1.5 rounds of 256 x 256 tiles), forward and backward: 1295 -> 1194 us, the forward 638 -> 571; a
// whole number of rounds is level (4096 rows 2207, 2209), so the choice between the two is half_tiles' (xq_gemm.hip).
//  * Two blocks on a compute unit, 80 KB of LDS each: one's start and end (7 of 26 us) run beside the other's products.  Blocks that
//    carry several tiles, the next one's first loads requested before the last one's end, stayed in step with each other: 6 % slower.
//  * Stages: three of activations, shared by the four waves, two of weights (nvfp4: three, with their scales), each wave's 64 columns its
//    own and waited for by that wave alone.  One barrier a K-step, three chunks before its end: behind it the first reads of the next K-step go out, so that nothing
//    waits at the seam.  Loads are in flight for 1.3 to 1.5 K-steps.
//  * A wave issues in order: a scalar or LDS-base instruction costs it as much as a vector one, and what does not fit between two MFMAs
//    is time.  M0 is written three times a K-step (not per load: 5 % of the launch), fragments are waited for in pairs, the scale of a
//    128-k block is a lane of a register (v_readlane; as a load that the compiler knows of it waited for every load in flight), and two
//    vector instructions follow each MFMA (four together behind four: 2.5 % slower).
//  * The end of a tile takes no LDS: side-term operands come straight into registers during the last K-step, and 16-lane rows swapped
//    between two column tiles make 16-byte pieces of an output row (7.3 -> 2.4 us).
#pragma once

#include <type_traits>
#include <utility>

#include "xq_gemm_dtl.h"

namespace xq {

template <int FMT>
struct GeoBank {
    static constexpr bool F4 = FMT == XQ_FMT_NVFP4;
    static constexpr int ROWS = 128, COLS = 256, BK = 64, NT = 256, NA = 3, NWS = F4 ? 3 : 2;
    static constexpr int A_BYTES = ROWS * BK * 2, W_BYTES = COLS * BK / (F4 ? 2 : 1), S_BYTES = F4 ? COLS * BK / 16 : 0;     // of a stage
    static constexpr size_t lds_bytes() { return (size_t)NA * A_BYTES + NWS * (W_BYTES + S_BYTES); }
};

// LDS instructions that chunk c of a K-step issues after its MFMAs, in this order: activation reads, weight reads (and their scales)
constexpr int bank_a_reads(int c, bool more) { return c <= 10 ? 1 : (more && c >= 13) ? (c < 15 ? 2 : 1) : 0; }
template <int FMT, bool CC>
constexpr int bank_w_reads(int c, bool more) {
    if (!more || c < 5 || c > 8) return 0;
    if (FMT == XQ_FMT_FP8) return CC ? 1 : 2;            // a weight tile
    return CC ? (c & 1) * 2 : 2;                         // CC: a pair of tiles and its scales every other chunk
}
// ... that are newer than chunk p's when chunk c begins
template <int FMT, bool CC>
constexpr int bank_newer_than_chunk(int p, int c, bool more) {
    int n = 0;
    for (int i = p + 1; i < c; ++i) n += bank_a_reads(i, more) + bank_w_reads<FMT, CC>(i, more);
    return n;
}
// ... and that are newer than the read of chunk c's activation fragment when chunk `at` begins
template <int FMT, bool CC>
constexpr int bank_newer(int c, int at, bool more) {
    // the fragment of chunk c: read in chunk c - 5, or (c < 5) behind the barrier of the K-step before: 0, 1 | 2, 3 | 4
    if (c < 5) return 4 - c + bank_newer_than_chunk<FMT, CC>(-1, at, more);
    return bank_w_reads<FMT, CC>(c - 5, more) + bank_newer_than_chunk<FMT, CC>(c - 5, at, more);
}

template <typename F, int... C>
__device__ __forceinline__ void bank_for_chunks(F&& chunk, std::integer_sequence<int, C...>) { (chunk(std::integral_constant<int, C>{}), ...); }

// two nvfp4 bytes of a dword (from byte B on), a column's four values of one scale -> 4 bf16
template <int B>
__device__ __forceinline__ u32x2 bank_decode4_f4(uint32_t w, float s) {
    const f32x2 a = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, B), b = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, B + 1);
    return u32x2{pack_bf16x2(a[0] * s, a[1] * s), pack_bf16x2(b[0] * s, b[1] * s)};
}

// two bytes' columns of a pair of nvfp4 weight tiles (its even and odd rows): word W of their operands
template <int W>
__device__ __forceinline__ void bank_pair_unit(uint32_t codes, uint32_t scales, float gs, u32x4& even, u32x4& odd) {
    constexpr int B = 2 * (W & 1);
    const f32x2 s = e4m3x2_to_f32(scales, B != 0);
    const f32x2 a = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(codes, 1.0f, B), b = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(codes, 1.0f, B + 1);
    const float s0 = s[0] * gs, s1 = s[1] * gs;
    even[W] = pack_bf16x2(a[0] * s0, b[0] * s1);
    odd[W] = pack_bf16x2(a[1] * s0, b[1] * s1);
}

template <int FMT, bool CC, bool DENSE = false>
__global__ void __launch_bounds__(256, 2) gemm_bank_kernel(G256Args g) {
    using D = GeoBank<FMT>;
    constexpr bool F4 = D::F4;
    constexpr int TM = 8, TN = 4, NC = 16;
    extern __shared__ __attribute__((aligned(16))) unsigned char dsm[];
    const int tid = threadIdx.x, lane = tid & 63, wn = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lg = lane >> 4;

    // ---- the tile and its expert: every wave counts the experts whose tiles end at or before this one
    int pid_m, pid_n, e = 0;
    if constexpr (DENSE) {
        const int nb = g.tiles_m * g.tiles_n, b = blockIdx.x, per = nb >> 3;
        const int logical = (b < per * 8) ? (b & 7) * per + (b >> 3) : b;
        constexpr int GM = 8;                                                 // row tiles beside each other: they share weight tiles
        const int width = GM * g.tiles_n, grp = logical / width, first_m = grp * GM, gsz = min(g.tiles_m - first_m, GM), in = logical - grp * width;
        pid_m = __builtin_amdgcn_readfirstlane(first_m + in % gsz);
        pid_n = __builtin_amdgcn_readfirstlane(in / gsz);
    } else {
        int pv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) pv[i] = g.tile_prefix[min(i * 64 + lane + 1, g.num_experts)];
        const int nb = g.tile_prefix[g.num_experts] * g.tiles_n;
        const int b = blockIdx.x, per = nb >> 3;
        if (b >= nb) return;
        const int logical = (b < per * 8) ? (b & 7) * per + (b >> 3) : b;
        pid_m = __builtin_amdgcn_readfirstlane(logical / g.tiles_n);          // all column tiles of a row tile side by side: an XCD stays on one expert's matrix
        pid_n = __builtin_amdgcn_readfirstlane(logical - pid_m * g.tiles_n);
#pragma unroll
        for (int i = 0; i < 4; ++i) e += __popcll(__ballot(pv[i] <= pid_m && i * 64 + lane < g.num_experts));
        for (int t0 = 256; t0 < g.num_experts; t0 += 64) {
            const int t = t0 + lane;
            e += __popcll(__ballot(t < g.num_experts && g.tile_prefix[min(t + 1, g.num_experts)] <= pid_m));
        }
        e = __builtin_amdgcn_readfirstlane(e);
    }
    const int row0 = DENSE ? pid_m * D::ROWS : __builtin_amdgcn_readfirstlane(g.offsets[e] + (pid_m - g.tile_prefix[e]) * D::ROWS);
    const int row_end = DENSE ? (int)g.M : __builtin_amdgcn_readfirstlane(g.offsets[e + 1]);
    const int n0 = pid_n * D::COLS;
    int n0w = n0, bank_width = g.Nout;
    const uint8_t* Wb = g.W + (int64_t)e * g.packed_stride;
    const uint8_t* Sb = g.scales + (int64_t)e * g.scale_stride;
    const uint8_t* Sb2 = g.W2 != nullptr ? g.scales2 + (int64_t)e * g.scale_stride : nullptr;
    const bf16_t* Ab = g.A;
    float gs = F4 ? g.global_scale[e] : 1.0f;
    const bf16_t* su_b = g.su;
    const bf16_t* lr_b = g.lora_right;
    // (dense: the second of two products of one shape on one input, gridDim.y; G256Args: W2, scales2, su2, bias2, right.f[1], and C from column
    // ncols1 on.  What differs is picked where it is used)
    const bool second_product = DENSE && blockIdx.y != 0;
    if (second_product) { Wb = g.W2; Sb = g.scales2; su_b = g.su2; }
    if constexpr (!DENSE && (!CC || F4)) {
        if (g.W2 != nullptr) {
            bank_width = g.ncols1;
            if (n0 >= g.ncols1) {
                Wb = g.W2 + (int64_t)e * g.packed_stride; Sb = Sb2; su_b = g.su2; lr_b = g.lora_right2; n0w = n0 - g.ncols1;
                Ab += g.a_off2;
                if (F4) gs = g.global_scale2[e];
            }
        }
    }
    const int nk = g.Kc / D::BK;
    const int scols = (g.wcols + 127) >> 7;
    // 16-row tiles that hold rows of the expert: the MFMAs of the others are skipped
    const int mt = __builtin_amdgcn_readfirstlane(min(TM, (row_end - row0 + 15) >> 4));

    // ---- direct-to-LDS sources: (a base every lane shares) + (a 32-bit byte offset of the lane's own).  A wave brings in 32
    // activation rows for the block, and the weights of its own 64 columns.
    constexpr int WP = F4 ? 2 : 4;                                    // its weight loads
    uint32_t a_off[4], w_off[WP], s_off = 0;
#pragma unroll
    for (int q = 0; q < WP; ++q) {
        if (F4 && CC) {                                               // 32 rows of bytes, a byte two output columns
            const int p = q * 16 + (lane >> 2);
            w_off[q] = (uint32_t)(min((n0w + wn * 64) / 2 + p, g.wrows / 2 - 1) * (int64_t)g.wcols + (((lane & 3) ^ ((p >> 2) & 2)) << 4)) + (3 - q) * 1024;
        } else if (F4) {                                              // 32 rows of bytes, a byte two k
            const int p = q * 16 + (lane >> 2), f = ((p >> 2) & 1) | (((p >> 3) & 1) << 1);
            w_off[q] = (uint32_t)((int64_t)p * g.wcols + min(n0w + wn * 64 + (((lane & 3) ^ f) << 4), g.wcols - 16)) + (3 - q) * 1024;
        } else if (CC) {
            const int rt = q * 16 + (lane >> 2);
            w_off[q] = (uint32_t)(min(n0w + wn * 64 + rt, g.wrows - 1) * (int64_t)g.wcols + (((lane & 3) ^ ((rt >> 2) & 2)) << 4)) + (3 - q) * 1024;
        } else {
            const int kr = q * 16 + (lane >> 2), f = ((kr >> 2) & 1) | (((kr >> 4) & 1) << 1);
            w_off[q] = (uint32_t)((int64_t)kr * g.wcols + min(n0w + wn * 64 + (((lane & 3) ^ f) << 4), g.wcols - 16)) + (3 - q) * 1024;
        }
    }
    // nvfp4 scales, [4][64] bytes: CC the four 16-column groups by k, !CC the four 16-k groups by column
    if (F4 && CC) s_off = (uint32_t)(min((n0w + wn * 64) / 16 + lg, g.wrows / 16 - 1) * (int64_t)g.wcols + l16 * 4);
    if (F4 && !CC) s_off = (uint32_t)((int64_t)lg * g.wcols + min(n0w + wn * 64 + l16 * 4, g.wcols - 4));
    const int64_t w_kstep = CC ? D::BK : (int64_t)(D::BK / (F4 ? 2 : 1)) * g.wcols, s_kstep = CC ? D::BK : 4 * (int64_t)g.wcols;
    const int nk1 = (!DENSE && !F4 && CC && g.W2 != nullptr) ? g.nk1 : (1 << 30);
    const int64_t w_jump = (!DENSE && !F4 && CC && g.W2 != nullptr) ? (g.W2 - g.W) - (int64_t)(nk1 - 1) * w_kstep : 0;      // to the second bank's first K-step
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)dsm;
    const uint32_t lds_w = lds0 + D::NA * D::A_BYTES + wn * (D::W_BYTES / 4);        // this wave's columns of weight stage 0
    // (M0, the LDS base of the loads, is written here and used nowhere else in the kernel: once for a run of parts, whose places in
    // LDS follow from the instruction's offset.  That offset counts on the global side too, so a lane's own offset is smaller by it,
    // and the base by 3 KB, to keep it positive.  The statement that writes M0 is not the one that reads it: the build refuses this kernel if
    // the compiler touches M0 by itself.)
    const uint32_t lds_s = lds0 + D::NA * D::A_BYTES + D::NWS * D::W_BYTES + wn * (D::S_BYTES / 4);
    const unsigned char* a_base = (const unsigned char*)Ab - 3072;
    const unsigned char* w_base = Wb - 3072;
    const unsigned char* s_base = Sb;
    auto begin_a = [&](int stage) { asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" :: "s"(lds0 + stage * D::A_BYTES + wn * 4096)); };
    auto begin_w = [&](int stage) { asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" :: "s"(lds_w + stage * D::W_BYTES)); };
#define XQ_BANK_ISSUE(off, base, p) asm volatile("global_load_lds_dwordx4 %0, %1 offset:%2" :: "v"(off[p]), "s"(base), "n"((p) * 1024) : "memory")
    auto next_a = [&]() { a_base += D::BK * 2; };
    auto next_w = [&](int kt) { w_base += !DENSE && !F4 && CC && kt == nk1 ? w_jump : w_kstep; };       // to K-step kt
    auto issue_s = [&](int stage) {                                    // four bytes a lane; then to the next K-step's
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" :: "s"(lds_s + stage * D::S_BYTES), "v"(s_off), "s"(s_base) : "memory");
        s_base += s_kstep;
    };
    int rows_src[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        rows_src[p] = min(row0 + (wn * 4 + p) * 8 + (lane >> 3), row_end - 1);
        if (!DENSE && g.a_rows) rows_src[p] = g.a_rows[rows_src[p]];
    }
    // block scales of this wave's columns: 128-k block kb in lane kb % 64, 64 blocks at a time
    const int sn = n0w + (wn >> 1) * 128;
    // (load and wait written out: a load that the compiler knows of would have it wait for every load in flight where the scale is used)
    auto load_scales = [&](int kb0) {
        const int kb = min(kb0 + lane, (nk - 1) >> 1);
        const bool second = !DENSE && 2 * kb >= nk1;                      // (nk1 is even: the matrices change on a scale-block boundary)
        const float* sp = (const float*)(second ? Sb2 : Sb);
        const int kb1 = second ? kb - (nk1 >> 1) : kb;
        const float* at = CC ? sp + (min(sn, g.wrows - 1) >> 7) * scols + kb1 : sp + (int64_t)kb1 * scols + (min(sn, g.wcols - 1) >> 7);
        float v;
        asm volatile("global_load_dword %0, %1, off\n\ts_waitcnt vmcnt(0)" : "=v"(v) : "v"(at) : "memory");
        return v;
    };
    float scales = F4 ? 0.0f : load_scales(0);
    auto scale_of = [&](int kt) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(scales), (kt >> 1) & 63)); };

#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const int rt = (wn * 4 + p) * 8 + (lane >> 3);
        a_off[p] = (uint32_t)((rows_src[p] * g.lda + (((lane & 7) ^ ((rt >> 1) & 5)) << 3)) * 2) + (3 - p) * 1024;
    }
#pragma unroll
    for (int st = 0; st < 2; ++st) {
        if (st) { next_w(1); next_a(); }
        begin_w(st);
        XQ_BANK_ISSUE(w_off, w_base, 0); XQ_BANK_ISSUE(w_off, w_base, 1);
        if constexpr (!F4) { XQ_BANK_ISSUE(w_off, w_base, 2 % WP); XQ_BANK_ISSUE(w_off, w_base, 3 % WP); }
        if constexpr (F4) issue_s(st);
        begin_a(st);
        XQ_BANK_ISSUE(a_off, a_base, 0); XQ_BANK_ISSUE(a_off, a_base, 1); XQ_BANK_ISSUE(a_off, a_base, 2); XQ_BANK_ISSUE(a_off, a_base, 3);
    }

    // ---- fragment reads, with the waits counted by hand (as in gemm_dtl16_kernel; no other LDS access inside the loop)
    uint32_t a_addr[2];
#pragma unroll
    for (int s_ = 0; s_ < 2; ++s_) a_addr[s_] = lds0 + l16 * 128 + ((((lg << 1) + s_) ^ ((l16 >> 1) & 5)) << 4);
    // (!CC: column tile j's chunk of 16 columns lies at this address with its bits 4 and 5 turned by j)
    const uint32_t w_addr = F4 && !CC ? lds_w + ((lg << 3) + (l16 >> 1)) * 64 + (((l16 >> 3) | ((lg & 1) << 1)) << 4) + ((l16 & 1) << 3)
                               : CC ? lds_w + l16 * 64 + ((lg ^ ((l16 >> 2) & 2)) << 4)
                               : lds_w + ((lg << 4) + (l16 >> 1)) * 64 + (((l16 >> 3) | ((lg & 1) << 1)) << 4) + ((l16 & 1) << 3);
#define XQ_BANK_READ_A(dst, so, c)                                                                                  \
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(a_addr[(c) / TM] + (so)), "n"(((c) % TM) * 2048))
    // nvfp4 scales.  !CC: column tile j's, of this lane's column and k group, a byte; CC: tile pair q's, of this lane's 16 k, 16 bytes
    const uint32_t s_addr = CC ? lds_s + (l16 >> 3) * 64 + lg * 16 : lds_s + lg * 64 + l16;
#define XQ_BANK_READ_W(j, wo, so)                                                                                  \
    do {                                                                                                            \
        if constexpr (F4 && CC) {                                                                                   \
            if constexpr ((j) % 2 == 0) {                                                                           \
                asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(raw[j]) : "v"(w_addr + (wo)), "n"((j) * 512));  \
                asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(raw[(j) + 1]) : "v"(s_addr + (so)), "n"((j) * 64)); \
            }                                                                                                       \
        } else if constexpr (F4) {                                                                                  \
            asm volatile("ds_read_b64_tr_b8 %0, %1" : "=v"(codes[j]) : "v"((w_addr + (wo)) ^ ((j) << 4)));          \
            asm volatile("ds_read_u8 %0, %1 offset:%2" : "=v"(sbyte[j]) : "v"(s_addr + (so)), "n"((j) * 16));       \
        } else if constexpr (CC) {                                                                                  \
            asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(raw[j]) : "v"(w_addr + (wo)), "n"((j) * 1024));     \
        } else {                                                                                                    \
            u32x2 lo_, hi_;                                                                                         \
            asm volatile("ds_read_b64_tr_b8 %0, %1" : "=v"(lo_) : "v"((w_addr + (wo)) ^ ((j) << 4)));               \
            asm volatile("ds_read_b64_tr_b8 %0, %1 offset:512" : "=v"(hi_) : "v"((w_addr + (wo)) ^ ((j) << 4)));    \
            raw[j] = u32x4{lo_[0], lo_[1], hi_[0], hi_[1]};                                                         \
        }                                                                                                           \
    } while (0)

    // (whole tiles have a copy of their own from here on, which carries no test of the row tiles)
    auto tile = [&](auto SKIP_) {
    constexpr bool SKIP = decltype(SKIP_)::value;
    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    bf16x8 fa[8];                 // ring: chunk c uses fa[c & 7]
    u32x4 fb0[TN], fb1[TN];       // decoded weight operands of step 0 / step 1 (8 bf16 each)
    u32x4 raw[TN];                // codes of the weight tiles (nvfp4, CC: of the pairs of tiles 0, 1 and 2, 3, each with its scales behind it)
    u32x2 codes[TN];              // nvfp4, !CC: the same, and their scales
    uint32_t sbyte[TN];
    float sv[TN], sv_next[TN], sc = 0.0f, sc_next = 0.0f;
    // operand words of a K-step's first 32 k from its codes, in eight units
    const auto first_unit = [&](auto U_) {
        constexpr int u = decltype(U_)::value, j = u >> 1, h = u & 1;
        if constexpr (F4 && CC) {
            constexpr int q = u >> 2, w = u & 3;
            bank_pair_unit<w>(raw[2 * q][w >> 1], raw[2 * q + 1][w >> 1], gs, fb0[2 * q], fb0[2 * q + 1]);
        } else {
            u32x2 d;
            if constexpr (F4) {
                if constexpr (h == 0) sv_next[j] = e4m3_to_f32((uint8_t)sbyte[j]) * gs;
                d = bank_decode4_f4<2 * h>(codes[j][0], sv_next[j]);
            } else {
                d = dtl_decode4(raw[j][h], sc_next);
            }
            fb0[j][2 * h] = d[0];
            fb0[j][2 * h + 1] = d[1];
        }
    };
    // the weights of K-step 0 have landed when only the loads behind them are still out
    if constexpr (F4) asm volatile("s_waitcnt vmcnt(11)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
    XQ_BANK_READ_W(0, 0u, 0u); XQ_BANK_READ_W(1, 0u, 0u); XQ_BANK_READ_W(2, 0u, 0u); XQ_BANK_READ_W(3, 0u, 0u);
    if constexpr (F4 && !CC)
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(codes[0]), "+v"(codes[1]), "+v"(codes[2]), "+v"(codes[3]), "+v"(sbyte[0]), "+v"(sbyte[1]),
                     "+v"(sbyte[2]), "+v"(sbyte[3]) :: "memory");
    else
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(raw[0]), "+v"(raw[1]), "+v"(raw[2]), "+v"(raw[3]) :: "memory");
    next_w(2);
    if constexpr (!F4) {
        begin_w(0);
        XQ_BANK_ISSUE(w_off, w_base, 0); XQ_BANK_ISSUE(w_off, w_base, 1);
        sc_next = scale_of(0);
    }
    bank_for_chunks(first_unit, std::make_integer_sequence<int, 8>{});
    // ... and the activations of K-step 0
    if constexpr (F4) asm volatile("s_waitcnt vmcnt(7)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(10)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    XQ_BANK_READ_A(fa[0], 0u, 0); XQ_BANK_READ_A(fa[1], 0u, 1); XQ_BANK_READ_A(fa[2], 0u, 2); XQ_BANK_READ_A(fa[3], 0u, 3); XQ_BANK_READ_A(fa[4], 0u, 4);

    // (the lane's place once more, for what follows the main loop: not kept in registers through it)
    int t16 = 0, tg = 0;
    // side term: operands of its first 32 ranks, requested while the last K-step's products run
    bf16x8 sx[TM], sw[TN];
    const int rp = g.r_pad;
    // (without a side term they are read from places that exist, and not used; whole tiles need no look at the rows' end)
    const unsigned char* su_t = (const unsigned char*)(rp > 0 ? su_b + (int64_t)row0 * g.ld_su : g.A);
    const unsigned char* lr_t = !DENSE && rp > 0 ? (const unsigned char*)(lr_b + (int64_t)e * bank_width * rp) : g.W;
    auto side_chunk = [&](int ks) { return max(min(ks * 4 + tg, (rp >> 3) - 1), 0) * 8; };
    auto side_x = [&](int i, int ks) {
        const int r = SKIP ? min(i * 16 + t16, row_end - 1 - row0) : i * 16 + t16;
        return *(const bf16x8*)(su_t + (uint32_t)((r * (int)g.ld_su + side_chunk(ks)) * 2));
    };
    // (dense: the factor as it is, converted here, behind the main loop, while the other block of the compute unit runs; chunks that hold
    // no rank at all are not looked at)
    const int ranks = DENSE ? min(rp, (g.right.r + 7) & ~7) : rp;
    auto side_w = [&](int j, int ks) {
        if constexpr (DENSE)
            return __builtin_bit_cast(bf16x8, right_chunk(g.right, second_product, min(n0w + wn * 64 + j * 16 + t16, g.Nout - 1), min(ks * 4 + tg, (ranks >> 3) - 1)));
        const int n = min(n0w + wn * 64 + (F4 && CC ? (j >> 1) * 32 + 2 * t16 + (j & 1) : j * 16 + t16), bank_width - 1);
        return *(const bf16x8*)(lr_t + (uint32_t)((n * rp + side_chunk(ks)) * 2));
    };
    auto in_rank = [&](const bf16x8& v, int ks) {        // lanes of ranks beyond rp get zeros
        const u32x4 z = {0, 0, 0, 0};
        return __builtin_bit_cast(bf16x8, (ks * 4 + tg) * 8 < ranks ? __builtin_bit_cast(u32x4, v) : z);
    };

    int sa = 0;                   // the activation stage of this K-step
    auto iteration = [&](int kt, auto MORE_, auto LATER_, auto LAST3_) {
        // MORE: there is a K-step kt + 1; LATER: kt + 2; LAST3: kt + 3
        constexpr bool MORE = decltype(MORE_)::value, LATER = decltype(LATER_)::value, LAST3 = decltype(LAST3_)::value;
        const int sb = sa == D::NA - 1 ? 0 : sa + 1, sp = sb == D::NA - 1 ? 0 : sb + 1;
        const uint32_t so = (uint32_t)sa * D::A_BYTES, son = (uint32_t)sb * D::A_BYTES;
        const uint32_t won = (uint32_t)(F4 ? sb : (kt + 1) & 1) * D::W_BYTES, sson = (uint32_t)sb * D::S_BYTES;
        // what the second 32 k need: this K-step's scales, and codes whose registers the next K-step's take
        sc = sc_next;
        u32x2 raw2[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            if constexpr (F4 && !CC) { raw2[j][0] = codes[j][1]; sv[j] = sv_next[j]; }
            else raw2[j] = u32x2{raw[j][2], raw[j][3]};
        }
        if constexpr (MORE && !F4) {
            if (((kt + 1) & 127) == 0) scales = load_scales((kt + 1) >> 1);
            sc_next = scale_of(kt + 1);
        }
        const auto second_unit = [&](auto U_) {
            constexpr int u = decltype(U_)::value, j = u >> 1, h = u & 1;
            if constexpr (F4 && CC) {
                constexpr int q = u >> 2, w = u & 3;
                bank_pair_unit<w>(raw2[2 * q][w >> 1], raw2[2 * q + 1][w >> 1], gs, fb1[2 * q], fb1[2 * q + 1]);
            } else {
                u32x2 d;
                if constexpr (F4) d = bank_decode4_f4<2 * h>(raw2[j][0], sv[j]);
                else d = dtl_decode4(raw2[j][h], sc);
                fb1[j][2 * h] = d[0];
                fb1[j][2 * h + 1] = d[1];
            }
        };
        auto chunk = [&](auto C_) {
            constexpr int c = decltype(C_)::value, i = c % TM;
            if constexpr (c == 13 && MORE) {
                // the next K-step's activations are there in every wave (behind them only the loads of this iteration), and the reads
                // of this one's, and of the next one's weights, are done: both stages may be written again
                constexpr int own = LATER ? (F4 ? 7 : 8) : 0;
                if constexpr (F4 && !CC)
                    asm volatile("s_waitcnt vmcnt(%5) lgkmcnt(0)" : "+v"(fa[5]), "+v"(fa[6]), "+v"(fa[7]), "+v"(codes[3]), "+v"(sbyte[3]) : "n"(own) : "memory");
                else
                    asm volatile("s_waitcnt vmcnt(%4) lgkmcnt(0)" : "+v"(fa[5]), "+v"(fa[6]), "+v"(fa[7]), "+v"(raw[3]) : "n"(own) : "memory");
                __builtin_amdgcn_s_barrier();
                XQ_BANK_READ_A(fa[0], son, 0); XQ_BANK_READ_A(fa[1], son, 1);
            } else if constexpr (MORE && (c == 8 || c == 12 || (c == 10 && !(F4 && CC)))) {
                // (the weight tile, or pair, whose decode begins here was read in chunk p)
                constexpr int p = F4 && CC ? c / 2 + 1 : 5 + (c - 8) / 2, j = (c - 8) / 2;
                constexpr int n = bank_newer_than_chunk<FMT, CC>(p, c, MORE), m = bank_newer<FMT, CC>(c + 1, c, MORE);
                if constexpr (F4 && CC)
                    asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(fa[c & 7]), "+v"(fa[(c + 1) & 7]), "+v"(raw[j]), "+v"(raw[j + 1]) : "n"(n < m ? n : m));
                else if constexpr (F4)
                    asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(fa[c & 7]), "+v"(fa[(c + 1) & 7]), "+v"(codes[j]), "+v"(sbyte[j]) : "n"(n < m ? n : m));
                else
                    asm volatile("s_waitcnt lgkmcnt(%3)" : "+v"(fa[c & 7]), "+v"(fa[(c + 1) & 7]), "+v"(raw[j]) : "n"(n < m ? n : m));
            } else if constexpr (!(MORE && c > 13)) {
                // (for two chunks at once)
                if constexpr (c % 2 == 0) asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(fa[c & 7]), "+v"(fa[(c + 1) & 7]) : "n"(bank_newer<FMT, CC>(c + 1, c, MORE)));
            }
            int rows_here = mt;
            if (SKIP) asm volatile("" : "+s"(rows_here));            // (compared in scalar registers, where it is used)
            if (!SKIP || i < rows_here)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, c < TM ? fb0[j] : fb1[j]), fa[c & 7], acc[i][j], 0, 0, 0);
            if constexpr (c <= 10) XQ_BANK_READ_A(fa[(c + 5) & 7], so, c + 5);
            if constexpr (MORE && c == 14) { XQ_BANK_READ_A(fa[2], son, 2); XQ_BANK_READ_A(fa[3], son, 3); }
            if constexpr (MORE && c == 15) XQ_BANK_READ_A(fa[4], son, 4);
            if constexpr (MORE && c == 5) {
                // the next K-step's weights: behind them the activations requested after them, and this iteration's loads so far
                constexpr int own = LATER ? (F4 ? 9 : 11) : 4;
                asm volatile("s_waitcnt vmcnt(%0)" :: "n"(own) : "memory");
            }
            if constexpr (MORE && c >= 5 && c <= 8) {
                if constexpr (!(F4 && CC)) XQ_BANK_READ_W(c - 5, won, sson);
                else if constexpr (c % 2 == 1) XQ_BANK_READ_W(c - 5, won, sson);
            }
            // eight vector instructions of the decode beside four MFMAs: the second 32 k, then the next K-step's first
            if constexpr (c < TM) second_unit(std::integral_constant<int, c>{});
            else if constexpr (MORE) first_unit(std::integral_constant<int, c - TM>{});
            // the loads of K-step kt + 2, one a chunk (several at once hold up the wave that issues them)
            constexpr int ca = F4 ? 3 : 2;
            if constexpr (LATER && c < 2) {
                if constexpr (c == 0) begin_w(F4 ? sp : kt & 1);
                XQ_BANK_ISSUE(w_off, w_base, F4 ? c : (c + 2) % WP);
            }
            if constexpr (F4 && LATER && c == 2) { next_w(kt + 3); issue_s(sp); }
            if constexpr (LATER && c >= ca && c < ca + 4) {
                if constexpr (c == ca) { next_a(); begin_a(sp); }
                XQ_BANK_ISSUE(a_off, a_base, c - ca);
            }
            if constexpr (!F4 && LAST3 && c >= 14) {
                if constexpr (c == 14) { next_w(kt + 3); begin_w((kt + 1) & 1); }
                XQ_BANK_ISSUE(w_off, w_base, c - 14);
            }
            if constexpr (!DENSE && !MORE && c == 12)
#pragma unroll
                for (int j = 0; j < TN; ++j) sw[j] = side_w(j, 0);
            if constexpr (!MORE && c >= 12) {
                sx[2 * (c - 12)] = side_x(2 * (c - 12), 0);
                sx[2 * (c - 12) + 1] = side_x(2 * (c - 12) + 1, 0);
            }
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);      // an MFMA,
                __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);      // two vector instructions
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        bank_for_chunks(chunk, std::make_integer_sequence<int, NC>{});
        sa = sb;
    };
    {
        using Y = std::true_type;
        using N = std::false_type;
        int kt = 0;
        for (; kt + 3 < nk; ++kt) iteration(kt, Y{}, Y{}, Y{});
        iteration(kt, Y{}, Y{}, N{});
        iteration(++kt, Y{}, N{}, N{});
        int lv = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
        asm volatile("" : "+v"(lv));
        t16 = lv & 15; tg = lv >> 4;
        iteration(++kt, N{}, N{}, N{});
    }

    for (int ks = 0; ks * 32 < rp; ++ks) {
        if (ks > 0)
#pragma unroll
            for (int i = 0; i < TM; ++i) sx[i] = side_x(i, ks);
        if constexpr (DENSE) {
#pragma unroll
            for (int i = 0; i < TM; ++i) sx[i] = in_rank(sx[i], ks);
#pragma unroll
            for (int j = 0; j < TN; ++j) {                             // one at a time, for the registers
                // (... and the addresses of all four, which do not change with ks, are not worked out ahead and kept: that is three to
                // eight registers more than there are beside the sums)
                asm volatile("" : "+v"(t16), "+v"(tg));
                const bf16x8 w = in_rank(side_w(j, ks), ks);
#pragma unroll
                for (int i = 0; i < TM; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, sx[i], acc[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            continue;
        }
        if (ks > 0)
#pragma unroll
            for (int j = 0; j < TN; ++j) sw[j] = side_w(j, ks);
#pragma unroll
        for (int j = 0; j < TN; ++j) sw[j] = in_rank(sw[j], ks);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const bf16x8 ax = in_rank(sx[i], ks);
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(sw[j], ax, acc[i][j], 0, 0, 0);
        }
    }

    const bf16_t* bias = second_product ? g.bias2 : g.bias;
    if (DENSE && bias) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const u32x2 b = *(const u32x2*)(bias + min(n0 + wn * 64 + j * 16 + 4 * tg, g.Nout - 4));
            const f32x4 b4 = {__uint_as_float(b[0] << 16), __uint_as_float(b[0] & 0xffff0000u), __uint_as_float(b[1] << 16), __uint_as_float(b[1] & 0xffff0000u)};
#pragma unroll
            for (int i = 0; i < TM; ++i) acc[i][j] += b4;
        }
    }

    // ---- the finished tile.  A lane holds, per (i, j) tile, row 16 i + l16 and the columns 16 j + 4 lg .. + 4.  Two column tiles side
    // by side swap the odd 16-lane rows of the first with the even ones of the second: a lane then has eight columns in a row, and
    // a store instruction writes 64 bytes of 16 rows -- without a trip through LDS.
    const int col = n0 + wn * 64 + (F4 && CC ? tg * 8 : (tg & 1) * 16 + (tg >> 1) * 8);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int row = row0 + i * 16 + t16;
        bf16_t* dst = g.C + (int64_t)row * g.ldc + col + (second_product ? g.ncols1 : 0);
#pragma unroll
        for (int jp = 0; jp < TN / 2; ++jp) {
            const f32x4 u = acc[i][2 * jp], v = acc[i][2 * jp + 1];
            u32x4 out;
            if constexpr (F4 && CC) {                                  // (the two tiles hold alternate columns)
                out = u32x4{pack_bf16x2(u[0], v[0]), pack_bf16x2(u[1], v[1]), pack_bf16x2(u[2], v[2]), pack_bf16x2(u[3], v[3])};
            } else {
                const auto s0 = __builtin_amdgcn_permlane16_swap(pack_bf16x2(u[0], u[1]), pack_bf16x2(v[0], v[1]), false, false);
                const auto s1 = __builtin_amdgcn_permlane16_swap(pack_bf16x2(u[2], u[3]), pack_bf16x2(v[2], v[3]), false, false);
                out = u32x4{s0[0], s1[0], s0[1], s1[1]};
            }
            if (row < row_end && col + jp * 32 < g.Nout) *(u32x4*)(dst + jp * 32) = out;
        }
    }
    };
    if (row_end - row0 >= D::ROWS) tile(std::false_type{});
    else tile(std::true_type{});
#undef XQ_BANK_ISSUE
#undef XQ_BANK_READ_A
#undef XQ_BANK_READ_W
}

// (dense block-fp8: f.W2 with ncols1 > 0 is the weight of a second product)
int launch_bank(const G256Args& f, int fmt, bool cc, hipStream_t s, const char* who);

}  // namespace xq
