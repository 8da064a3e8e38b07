// Dense weights under many rows: the weight is decoded once into bf16 K-step images, and a kernel that does nothing but load,
// read and multiply runs over them.
//
//   C[rows, Nout] = A[rows, Kc] . Wop (+ su[rows, r] . Lr[Nout, r]^T) (+ bias)        Wop as in xq_gemm_256.h
//
// gemm_256_kernel decodes a 4-bit weight tile for every 256 rows: at 4096 rows each code is looked up 16 times, and the vector
// instructions of the decode and the LDS stores of its results hold the matrix pipes at 0.85-0.92 PFLOP/s; gemm_dtl16_kernel
// (block-fp8) decodes beside its MFMAs at 1.20-1.24.  Over an image the same tiles run at 1.30-1.38 PFLOP/s (nvfp4 [8192, 5120]
// under 4096 rows: 375 us before, 260 + 29 for the image; block-fp8 [12288, 4096] under 8192: 686, 600 + 26), held there by
// the power the matrix units draw on random operands.  The image costs one pass over the weight, at 4.5-5.8 TB/s of codes
// read and bf16 written.  Its values are the stand-alone decoders', bit for bit.
//  * Image.  [tile of 256 output columns][K-step of 32][256 n][32 k] bf16, 16 KB per K-step and tile; the 16-byte chunk c of row
//    n lies at chunk c ^ ((n >> 2) & 2), as the kernel wants it in LDS (the stage layout of gemm_dtl16_kernel's weight bytes:
//    its 16-byte reads meet no bank conflict), so a direct-to-LDS load is a copy of 1 KB in a row.  Forward and dgrad
//    write the same form (the dgrad's pass transposes), and one kernel serves both.  Columns beyond the matrix repeat the last.
//  * Kernel.  Tiles of 32 TM x 64 TN, K-steps of 32: 256 x 256 (TM 8, TN 4), 224, 288 or 320 rows, or 320 columns, by what fills the
//    chip's rounds best (plan_decoded, xq_gemm.hip).  Four LDS stages (activations in the same chunk order), eight waves of 16 TM x 16 TN
//    on v_mfma_f32_16x16x32_bf16.  A K-step is TM chunks of TN MFMAs; the activation fragment of a chunk is read three chunks ahead,
//    the weight fragments of the next K-step during this one's first chunks (two register sets), the loads of K-step kt + 3 go
//    out one per chunk.  In iteration kt every wave reads stages kt and kt + 1 and writes stage kt + 3: the loads of kt + 2 are
//    waited for at its end (those of kt + 3 stay in flight), so a load has two iterations to land and no read waits behind the
//    barrier.
//  * Splits.  gridDim.y blocks divide the K-steps of a tile (pairs of them: every part is even) where tiles alone leave a
//    round of the chip part empty; each part writes its fp32 sums, splitk_reduce_kernel adds them.
#pragma once

#include "xq_gemm_dtl.h"

namespace xq {

struct GeoDec {
    static constexpr int T = 256, NT = 512, BK = 32, STAGES = 4;   // T: columns of an image tile
    static constexpr int TILE_BYTES = T * BK * 2;                  // a K-step of it: 16 KB
    static constexpr int MIN_STEPS = 4;                            // K-steps of a part (an even number)
};

// A block's tile: 32 TM rows x 64 TN columns
template <int TM, int TN>
struct GeoDecTile {
    static constexpr int ROWS = 32 * TM, COLS = 64 * TN;
    static constexpr int A_BYTES = ROWS * GeoDec::BK * 2, STAGE_BYTES = A_BYTES + COLS * GeoDec::BK * 2;
    static constexpr int AP = (ROWS / 8 + 15) / 16, WP = (COLS / 8 + 15) / 16;     // direct loads of a wave and K-step
    static constexpr size_t lds_bytes() { return (size_t)GeoDec::STAGES * STAGE_BYTES; }
};

inline int64_t dec_image_bytes(int64_t Nout, int64_t Kc) { return xq_cdiv(Nout, GeoDec::T) * GeoDec::T * Kc * 2; }

struct DecImageArgs {
    const uint8_t* packed;
    const uint8_t* scales;
    const float* global_scale;
    int32_t wrows, wcols, gshift, scale_dtype;
    int32_t Kc, Nout;       // of this matrix
    bf16_t* image;
    int32_t nk, kt0;        // K-steps of the image, and the first of them that this matrix fills (two matrices: one sum)
};


__device__ __forceinline__ int64_t dec_image_at(int64_t n, int kt, int nk, int chunk) {
    return (((n >> 8) * nk + kt) * 256 + (n & 255)) * 32 + ((chunk ^ (int)((n >> 2) & 2)) << 3);
}

// the sixteen NF4 levels in LDS (a per-lane index into constant memory is a vector load)
template <int FMT>
__device__ __forceinline__ float dec_val(uint32_t nib, float s, const float* levels) {
    if constexpr (FMT == XQ_FMT_NF4) return levels[nib] * s;
    else return val4<FMT>(nib, s);
}

// 8 consecutive codes of one scale (4-bit: the first dword, block-fp8: both) as the fp32 values the decoders round
template <int FMT>
__device__ __forceinline__ void dec8(float (&v)[8], u32x2 w, float s, const float* levels) {
    if constexpr (FMT == XQ_FMT_FP8) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const f32x2 lo = e4m3x2_to_f32(w[h], false), hi = e4m3x2_to_f32(w[h], true);
            v[4 * h] = lo[0] * s; v[4 * h + 1] = lo[1] * s; v[4 * h + 2] = hi[0] * s; v[4 * h + 3] = hi[1] * s;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = dec_val<FMT>((w[0] >> (4 * i)) & 0xfu, s, levels);
    }
}

// codes and scale of the 8 elements from row, col on (col % 8 == 0)
template <int FMT>
__device__ __forceinline__ void dec8_load(const DecImageArgs& g, int64_t row, int64_t col, u32x2* w, float* s) {
    const int64_t at = row * g.wcols + col;
    if constexpr (FMT == XQ_FMT_FP8) {
        *w = *(const u32x2*)(g.packed + at);
        *s = ((const float*)g.scales)[(row >> 7) * ((g.wcols + 127) >> 7) + (col >> 7)];
    } else {
        (*w)[0] = *(const uint32_t*)(g.packed + (at >> 1));
        *s = load_scale(g.scales, at >> g.gshift, g.scale_dtype);
    }
}

// CC (W [Nout, Kc]): a block takes 32 rows x 256 k, a thread 8 codes of four rows
template <int FMT>
__global__ void __launch_bounds__(256) dec_image_kernel(DecImageArgs g) {
    __shared__ float levels[16];
    if (FMT == XQ_FMT_NF4) {
        if (threadIdx.x < 16) levels[threadIdx.x] = kNf4Level[threadIdx.x];
        __syncthreads();
    }
    const int k = (blockIdx.x * 32 + (threadIdx.x & 31)) * 8;
    if (k >= g.Kc) return;
    const int64_t n0 = (int64_t)blockIdx.y * 32 + (threadIdx.x >> 5);
    const float gs = FMT == XQ_FMT_NVFP4 ? g.global_scale[0] : 1.0f;
    u32x2 w[4];
    float s[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) dec8_load<FMT>(g, min(n0 + 8 * i, (int64_t)g.Nout - 1), k, &w[i], &s[i]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float v[8];
        dec8<FMT>(v, w[i], FMT == XQ_FMT_NVFP4 ? s[i] * gs : s[i], levels);
        *(u32x4*)(g.image + dec_image_at(n0 + 8 * i, g.kt0 + (k >> 5), g.nk, (k >> 3) & 3)) =
            u32x4{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
    }
}

// !CC (W [Kc, Nout]): a block takes 64 k x 256 columns, a thread 8 k x 8 columns
template <int FMT>
__global__ void __launch_bounds__(256) dec_image_t_kernel(DecImageArgs g) {
    __shared__ float levels[16];
    if (FMT == XQ_FMT_NF4) {
        if (threadIdx.x < 16) levels[threadIdx.x] = kNf4Level[threadIdx.x];
        __syncthreads();
    }
    const int kc = threadIdx.x & 7;
    const int k0 = blockIdx.x * 64 + kc * 8;
    const int64_t n0 = (int64_t)blockIdx.y * 256 + (threadIdx.x >> 3) * 8;
    const int64_t col = min(n0, (int64_t)g.Nout - 8);
    const float gs = FMT == XQ_FMT_NVFP4 ? g.global_scale[0] : 1.0f;
    u32x2 w[8];
    float s[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) dec8_load<FMT>(g, k0 + i, col, &w[i], &s[i]);
    uint32_t p[8][4];                       // [column][pair of k]
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float a[8], b[8];
        dec8<FMT>(a, w[2 * i], FMT == XQ_FMT_NVFP4 ? s[2 * i] * gs : s[2 * i], levels);
        dec8<FMT>(b, w[2 * i + 1], FMT == XQ_FMT_NVFP4 ? s[2 * i + 1] * gs : s[2 * i + 1], levels);
#pragma unroll
        for (int j = 0; j < 8; ++j) p[j][i] = pack_bf16x2(a[j], b[j]);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
        *(u32x4*)(g.image + dec_image_at(n0 + j, g.kt0 + (k0 >> 5), g.nk, kc & 3)) = u32x4{p[j][0], p[j][1], p[j][2], p[j][3]};
}

// G256Args::W is the image; ksplit and partial as there (SPLIT: fp32 sums to partial, part 0 with side term and bias)
template <bool SPLIT, int TM, int TN>
__global__ void __launch_bounds__(512, 2) gemm_dec_kernel(G256Args g) {
    using D = GeoDec;
    using G = GeoDecTile<TM, TN>;
    constexpr int NC = TM, NP = G::AP + G::WP, RW = TM * 16, CW = TN * 16;
    constexpr int RING = NC % 4 == 0 ? 4 : NC % 5 == 0 ? 5 : NC;       // activation fragments held: a divisor of the chunks, above 3
    static_assert(TN <= NC - 2 && NP <= NC, "the waits below");
    extern __shared__ __attribute__((aligned(16))) unsigned char dsm[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 2, wn = wave & 3;
    const int l16 = lane & 15, lg = lane >> 4;

    int pid_m, pid_n;
    {
        const int nb = g.tiles_m * g.tiles_n;
        const int b = blockIdx.x, per = nb >> 3;
        const int logical = (b < per * 8) ? (b & 7) * per + (b >> 3) : b;
        constexpr int GM = 4;
        const int width = GM * g.tiles_n;
        const int grp = logical / width, first_m = grp * GM;
        const int gsz = min(g.tiles_m - first_m, GM);
        const int in = logical - grp * width;
        pid_m = first_m + in % gsz;
        pid_n = in / gsz;
    }
    const int64_t row0 = (int64_t)pid_m * G::ROWS, row_end = g.M;
    const int n0 = pid_n * G::COLS;
    const int nk_all = g.Kc / D::BK;
    int kt0 = 0, nk = nk_all;                           // this part's K-steps: an even number, MIN_STEPS or more
    if constexpr (SPLIT) {
        const int pairs = nk_all >> 1, s = blockIdx.y;
        kt0 = 2 * (int)((int64_t)pairs * s / g.ksplit);
        nk = 2 * (int)((int64_t)pairs * (s + 1) / g.ksplit) - kt0;
    }
    const int mt = __builtin_amdgcn_readfirstlane((int)max((int64_t)0, min((int64_t)TM, (row_end - row0 - wm * RW + 15) >> 4)));

    // ---- direct-to-LDS sources: a wave brings in an eighth of the activation rows and of the image columns, 64 bytes of each, 16
    // to a load (the last load of either: what is left)
    uint32_t a_off[G::AP], w_off[G::WP];
#pragma unroll
    for (int p = 0; p < G::AP; ++p) {
        const int rt = wave * (G::ROWS / 8) + p * 16 + (lane >> 2);
        const int64_t r = min(row0 + rt, row_end - 1);
        a_off[p] = (uint32_t)((r * g.lda + (((lane & 3) ^ ((rt >> 2) & 2)) << 3)) * 2);
    }
    const int t0 = n0 >> 8;
#pragma unroll
    for (int p = 0; p < G::WP; ++p) {
        // (a tile that does not begin with an image tile lies across two; columns beyond the image: its last)
        const int n = min(n0 + wave * (G::COLS / 8) + p * 16 + (lane >> 2), (int)((g.Nout + 255) & ~255) - 1);
        w_off[p] = (uint32_t)((n >> 8) - t0) * (uint32_t)(nk_all * D::TILE_BYTES) + (uint32_t)(n & 255) * 64 + (lane & 3) * 16;
    }
    const unsigned char* const a_base = (const unsigned char*)(g.A + (int64_t)kt0 * D::BK);
    const unsigned char* const w_base = g.W + ((int64_t)t0 * nk_all + kt0) * D::TILE_BYTES;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)dsm;
    // (M0 as in gemm_dtl16_kernel: the LDS base of the load, written here and used nowhere else)
    auto issue_part = [&](int kt, int part) {
        const uint32_t stage = lds0 + (uint32_t)(kt & 3) * G::STAGE_BYTES;
        const bool of_a = part < G::AP;
        const int p = of_a ? part : part - G::AP, rows = (of_a ? G::ROWS : G::COLS) / 8;
        const uint32_t dst = stage + (of_a ? 0 : G::A_BYTES) + wave * rows * 64 + p * 1024;
        const unsigned char* base = of_a ? a_base + (int64_t)kt * (D::BK * 2) : w_base + (int64_t)kt * D::TILE_BYTES;
        const uint32_t off = of_a ? a_off[p] : w_off[p];
        if (p * 16 + 16 <= rows || lane < (rows - p * 16) * 4)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(dst), "v"(off), "s"(base) : "memory");
    };

    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // ---- fragment reads, with the waits counted by hand (as in gemm_dtl16_kernel; no other LDS access inside the loop).  To the
    // compiler a fragment is there with its read: were one spilled before its wait, what is stored would be what the register held
    // before.  Hence no spills here at all, which the build checks.
    const int sw = (l16 >> 2) & 2;
    const uint32_t a_addr = lds0 + (wm * RW + l16) * 64 + ((lg ^ sw) << 4);
    const uint32_t w_addr = lds0 + G::A_BYTES + (wn * CW + l16) * 64 + ((lg ^ sw) << 4);
#define XQ_DEC_READ(dst, addr, so, t) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"((addr) + (so)), "n"((t) * 1024))

    // ---- prologue: K-steps 0, 1 and 2 requested, 0 and 1 waited for
#pragma unroll
    for (int kt = 0; kt < 3; ++kt)
#pragma unroll
        for (int part = 0; part < NP; ++part) issue_part(kt, part);
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(NP) : "memory");
    __builtin_amdgcn_s_barrier();

    bf16x8 fa[RING];              // chunk c uses fa[c % RING]
    bf16x8 fb[2][TN];             // weight fragments of even and odd K-steps
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int j = 0; j < TN; ++j) XQ_DEC_READ(fb[0][j], w_addr, 0u, j);
    XQ_DEC_READ(fa[0], a_addr, 0u, 0); XQ_DEC_READ(fa[1], a_addr, 0u, 1); XQ_DEC_READ(fa[2], a_addr, 0u, 2);
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(fa[0]), "+v"(fa[1]), "+v"(fa[2]));
#pragma unroll
    for (int j = 0; j < TN; ++j) asm volatile("" : "+v"(fb[0][j]));

    // LDS reads that chunk c of an iteration issues (c < 0: of the iteration before, which had a next one)
    auto reads_in_chunk = [](int c, bool more) constexpr -> int {
        if (c < 0) return 1;                                            // its last two: one activation read each
        return (c + 3 < NC || more ? 1 : 0) + (more && c < TN ? 1 : 0);
    };
    auto iteration = [&](int kt, auto P_, auto LEFT_, auto SKIP_) {
        // LEFT: K-steps behind this one, 3 for "three or more"
        constexpr int P = decltype(P_)::value, LEFT = decltype(LEFT_)::value;
        constexpr bool MORE = LEFT >= 1, SKIP = decltype(SKIP_)::value;
        const uint32_t so = (uint32_t)(kt & 3) * G::STAGE_BYTES, son = (uint32_t)((kt + 1) & 3) * G::STAGE_BYTES;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            // the chunk's activation fragment (and, older, the K-step's weight fragments) have landed when only the reads of
            // the two chunks before are still out
            {
                const int n = reads_in_chunk(c - 1, MORE) + reads_in_chunk(c - 2, MORE);
                if (c == 0) {
                    asm volatile("s_waitcnt lgkmcnt(2)" : "+v"(fa[0]));
#pragma unroll
                    for (int j = 0; j < TN; ++j) asm volatile("" : "+v"(fb[P][j]));
                } else if (n == 1) asm volatile("s_waitcnt lgkmcnt(1)" : "+v"(fa[c % RING]));
                else if (n == 2) asm volatile("s_waitcnt lgkmcnt(2)" : "+v"(fa[c % RING]));
                else if (n == 3) asm volatile("s_waitcnt lgkmcnt(3)" : "+v"(fa[c % RING]));
                else if (n == 4) asm volatile("s_waitcnt lgkmcnt(4)" : "+v"(fa[c % RING]));
                else asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(fa[c % RING]));
            }
            if (!SKIP || c < mt)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[c][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[P][j], fa[c % RING], acc[c][j], 0, 0, 0);
            if (c + 3 < NC) XQ_DEC_READ(fa[(c + 3) % RING], a_addr, so, c + 3);
            else if (MORE) XQ_DEC_READ(fa[(c + 3) % RING], a_addr, son, c + 3 - NC);
            if (MORE && c < TN) XQ_DEC_READ(fb[P ^ 1][c], w_addr, son, c);
            if (LEFT >= 3 && c < NP) issue_part(kt + 3, c);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (MORE) {
            // the loads of K-step kt + 2 have landed
            if (LEFT >= 3) asm volatile("s_waitcnt vmcnt(%0)" :: "n"(NP) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    {
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
        using I2 = std::integral_constant<int, 2>;
        using I3 = std::integral_constant<int, 3>;
        auto run = [&](auto SKIP_) {
            int kt = 0;
            for (; kt + 4 < nk; kt += 2) {
                iteration(kt, I0{}, I3{}, SKIP_);
                iteration(kt + 1, I1{}, I3{}, SKIP_);
            }
        };
        if (mt == TM) run(std::false_type{});
        else run(std::true_type{});
        // the last four of either loop, once: behind each of them the sums met with no register to spare and some went to scratch
        const int kt = nk - 4;
        iteration(kt, I0{}, I3{}, std::true_type{});
        iteration(kt + 1, I1{}, I2{}, std::true_type{});
        iteration(kt + 2, I0{}, I1{}, std::true_type{});
        iteration(kt + 3, I1{}, I0{}, std::true_type{});
    }
#undef XQ_DEC_READ

    // (the lane read again: what the end needs of it is not kept through the loop)
    int lane_e;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(lane_e));
    const int tid_e = wave * 64 + lane_e;
    if constexpr (SPLIT) {
        const int s = blockIdx.y;
        G256Args f = g;
        if (s > 0) { f.r_pad = 0; f.bias = nullptr; }
        dtl16_side_term<TM, TN>(f, dsm, G::ROWS * 128, acc, row0, row_end, n0, tid_e);
        float* part = g.partial + (int64_t)s * g.M * g.Nout;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = n0 + wn * CW + j * 16 + 4 * (lane_e >> 4);
            f32x4 b4 = {0.0f, 0.0f, 0.0f, 0.0f};
            if (f.bias) {
                const u32x2 b = *(const u32x2*)(f.bias + min(n, g.Nout - 4));
                b4 = f32x4{__uint_as_float(b[0] << 16), __uint_as_float(b[0] & 0xffff0000u), __uint_as_float(b[1] << 16), __uint_as_float(b[1] & 0xffff0000u)};
            }
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int64_t row = row0 + wm * RW + i * 16 + (lane_e & 15);
                if (row < row_end && n < g.Nout) *(f32x4*)(part + row * g.Nout + n) = acc[i][j] + b4;
            }
        }
    } else {
        dtl16_finish<TM, TN>(g, dsm, G::ROWS * 128, acc, row0, row_end, n0, tid_e);
    }
}

}  // namespace xq
