// Merging the LoRA update into the quantized base weight without materialising it:
//
//   W'[n, k] = deq(W)[n, k] + scaling * sum_j B[n, j] * A[j, k]          (W FLAT [N, K])
//
// A block owns 128 x 128 tiles, each exactly one block-fp8 scale block: a run of them down a strip of 128 columns, so that the strip's
// columns of A are split once for all of them and the next tile's codes and rows of B are in flight while one is worked on.  Per tile it
//   1. computes the low-rank product on the matrix cores.  The reference multiplies the fp32 factors in fp32; here each factor is
//      split into two bf16 terms (hi + lo, 16 significant bits) and the product is the three bf16 MFMA products hi*hi + hi*lo +
//      lo*hi with fp32 accumulation (relative error ~2^-16 per term instead of 2^-9 with plain bf16 factors).  The factors are read as
//      they are stored (as many bytes in fp32 as the two bf16 parts have) and split on the way to LDS;
//   2. hands it to the row-contiguous pass through LDS: every thread decodes runs of 16 columns, whole 128-byte lines of codes
//      being read by neighbouring lanes, to the reference decoder's value and adds the update;
//   3a. (publish) rounds to bf16 -- bf16(bf16(deq) + bf16(delta)), the arithmetic of the reference's
//      weight-sync merge -- or writes the fp32 sum; or
//   3b. (requantise, block-fp8) reduces the tile's absmax, derives the new block scale
//      s = max(amax / 448, 1e-12) and writes e4m3(clamp(x / s)) bytes and the scale: decode -> add ->
//      re-encode in one pass over 1 byte per weight each way; or
//   3c. (requantise, 4-bit) encodes the published values, whose groups are the runs of one, four or eight neighbouring lanes.
#include "xq_common.h"
#include "xq_codes.h"
#include <atomic>
#include "xq_lora.h"

namespace xq {

constexpr int MG_T = 128;           // tile edge
// Blocks of a launch at most: two a CU, what the registers (128 a lane) and LDS (74 KB) allow at once, so that every block takes an
// equal run of tiles.  With 1024, 1536 and a block per tile instead, [12288, 4096] r 32, us: int4 publish 37.7 -> 40.0, 40.9, 45.1;
// nvfp4 requantise 86.8 -> 90.2, 94.9, 108.6; block-fp8 requantise 31.6 -> 33.7, 34.9, 39.1; [8192, 5120] nf4 34.5 -> 40.0, 39.8, 39.4.
constexpr int MG_BLOCKS = 2 * 256;

struct MergeArgs {
    const uint8_t* packed;
    const uint8_t* scales;
    const float* global_scale;
    int32_t fmt, group, scale_dtype;
    int32_t N, K;
    const void* A;       // [r, K]
    const void* B;       // [N, r]
    int32_t lora_f32, r, r_pad;
    float scaling;
    int32_t run;         // merge_tiles
    int32_t mode;        // 0: bf16 out (publish arithmetic), 1: fp32 out, 2: block-fp8 requantise,
                         // 3: absmax of the mode-0 values only, 4 / 5: nvfp4 / nf4 requantise of the mode-0 values,
                         // 6 / 7: int4 requantise of the mode-0 values, 128-element groups along K (6: scale =
                         // bf16(absmax / 7), codes rne(x / scale) in [-7, 7] + 8; 7: the reference's rule, fp32 scales)
    void* out;           // mode 0/1: [N, K]
    uint8_t* packed_out; // mode 2: [N, K] e4m3 bytes    } both may alias the inputs: a block reads its tile and its
    float* scales_out;   // mode 2: [ceil(N/128), ceil(K/128)] } scale before it writes them, and touches no other
                         // mode 5: [N, K/64] fp32; mode 6: [N, K/128] bf16; mode 7: [N, K/128] fp32
    float* amax_out;     // mode 3: one float, zeroed before the launch; receives max |value| over the matrix
    const float* gamax;  // mode 4: the tensor-level amax the scales are derived from (one float on the device)
    uint8_t* codes_out;  // mode 4 / 5: [N, K/2] code pairs     } may alias the inputs (tile-local, read before written);
    uint8_t* bscale_out; // mode 4: [N, K/16] e4m3 block scales } the global scale output may not
    float* gscale_out;   // mode 4: one float
};

__device__ __forceinline__ void lds_barrier() {       // (leaves loads in flight)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// max over the 64 lanes of values >= 0, in lane 63 (six vector instructions; through LDS, as __shfl_xor goes, it is six round trips)
__device__ __forceinline__ float wave_max63(float v) {
#define XQ_DPP(CTRL) v = fmaxf(v, __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), CTRL, 0xf, 0xf, true)))
    XQ_DPP(0x111); XQ_DPP(0x112); XQ_DPP(0x114); XQ_DPP(0x118);         // row_shr:1, 2, 4, 8
    XQ_DPP(0x142); XQ_DPP(0x143);                                       // row_bcast:15, 31
#undef XQ_DPP
    return v;
}

// A block's tiles, counted down the strips: run > 0, that many of one strip, neighbouring blocks at the same height of neighbouring
// strips; otherwise an equal share of all
__device__ __forceinline__ void merge_tiles(int run, uint32_t tiles_n, uint32_t tiles_k, int64_t& first, int64_t& last, int& nt, int& kt) {
    if (run > 0) {
        kt = (int)(blockIdx.x % tiles_k);
        nt = (int)(blockIdx.x / tiles_k) * run;
        first = (int64_t)kt * tiles_n + nt;
        last = first + (run < (int)tiles_n - nt ? run : (int)tiles_n - nt);
    } else {
        const int64_t total = (int64_t)tiles_n * tiles_k;
        first = total * blockIdx.x / gridDim.x;
        last = total * (blockIdx.x + 1) / gridDim.x;
        kt = (int)(first / tiles_n);
        nt = (int)(first - (int64_t)kt * tiles_n);
    }
}

// 16 bytes from any factor element on (one global_load_dwordx4 like an aligned one)
typedef u32x4 u32x4_a2 __attribute__((aligned(2)));

// Eight factor elements as they are stored -> their hi and lo bf16 parts, times `by`; ranks from g.r on are zero.  pairs: two bf16 to
// a word
__device__ __forceinline__ void merge_split8(const MergeArgs& g, const uint32_t (&raw)[8], bool pairs, float by, int j0, u32x4& hi, u32x4& lo) {
    float f[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const uint32_t bits = g.lora_f32 ? raw[e] : !pairs ? raw[e] << 16 : e & 1 ? raw[e >> 1] & 0xffff0000u : raw[e >> 1] << 16;
        f[e] = j0 + e < g.r ? __uint_as_float(bits) * by : 0.0f;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        hi[e] = pack_bf16x2(f[2 * e], f[2 * e + 1]);
        lo[e] = pack_bf16x2(f[2 * e] - __uint_as_float(hi[e] << 16), f[2 * e + 1] - __uint_as_float(hi[e] & 0xffff0000u));
    }
}

// The factors of a tile of 512 threads.  In LDS: [hi, lo][128][RP + 8], which reads and writes without bank conflicts.
template <int RP>
struct MergeFactors {
    static constexpr int FP = RP + 8, R8 = RP > 0 ? RP / 8 : 1, KS = RP / 16;
    static constexpr int BYTES = 2 * MG_T * FP * 2;
    static constexpr int NB = (RP + 31) / 32, ITEMS = 16 * RP;         // B: eight ranks of a row an item
    uint32_t raw[NB > 0 ? NB : 1][8];

    // a thread's item i.  Where R8 is no power of two (RP 48) its row and piece are formed per tile, behind the empty statement, not kept
    // through the loop: every kernel of that rank spilled for them, up to 29 registers a lane (absmax at r 40, [12288, 4096]: 45 us,
    // without 42)
    static __device__ __forceinline__ int item(int tid, int i) {
        int b = tid + 512 * i;
        if constexpr ((R8 & (R8 - 1)) != 0) asm volatile("" : "+v"(b));
        return b;
    }
    // the tile's rows of B -> registers, as they are stored (clamped to the last row).  Eight ranks are one or two 16-byte loads at whatever
    // address the first of them has; what these read past the end of a row the split zeroes, and only where it would lie past the
    // matrix are the elements loaded one by one.  The branches on the type go around the loads: one between them, for a value that
    // either type writes, makes the second wait for the first.  [12288, 4096], us, with 16-byte loads for multiples of 8 only and that
    // branch -> now: block-fp8 requantise r 63 55.6 -> 42.7, r 64 43.6 -> 42.7; publish r 63 62.0 -> 45.3, r 40 44.0 -> 42.0; nf4 requantise
    // r 63 76.6 -> 62.5, r 16 48.6 -> 44.4.
    __device__ __forceinline__ void load_b(const MergeArgs& g, int n0, int tid, int wave) {
        const int64_t end = (int64_t)g.N * g.r;
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int b = item(tid, i);
            if (512 * i + 512 > ITEMS && 512 * i + wave * 64 >= ITEMS) break;
            const int nb = n0 + b / R8, j0 = b % R8 * 8;
            const int64_t at = (int64_t)(nb < g.N ? nb : g.N - 1) * g.r + (j0 < g.r ? j0 : 0);
            const int last = (int)(end - at < 8 ? end - at : 8) - 1;        // of the eight, the last within the matrix
            if (g.lora_f32) {
                const uint32_t* p = (const uint32_t*)g.B + at;
                if (last == 7) {
                    const u32x4 lo = *(const u32x4_a2*)p, hi = *(const u32x4_a2*)(p + 4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) { raw[i][e] = lo[e]; raw[i][4 + e] = hi[e]; }
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e) raw[i][e] = p[e < last ? e : last];
                }
            } else {
                const uint16_t* p = (const uint16_t*)g.B + at;
                if (last == 7) {
                    const u32x4 lo = *(const u32x4_a2*)p;
#pragma unroll
                    for (int e = 0; e < 4; ++e) { raw[i][e] = lo[e]; raw[i][4 + e] = 0u; }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        raw[i][e] = p[2 * e < last ? 2 * e : last] | (uint32_t)p[2 * e + 1 < last ? 2 * e + 1 : last] << 16;
                        raw[i][4 + e] = 0u;
                    }
                }
            }
        }
    }
    __device__ __forceinline__ void store_b(const MergeArgs& g, bf16_t* sh_b, int tid, int wave) const {
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int b = item(tid, i);
            if (512 * i + 512 > ITEMS && 512 * i + wave * 64 >= ITEMS) break;
            u32x4 hi, lo;
            merge_split8(g, raw[i], true, g.scaling, b % R8 * 8, hi, lo);
            bf16_t* to = sh_b + b / R8 * FP + b % R8 * 8;
            *(u32x4*)to = hi;
            *(u32x4*)(to + MG_T * FP) = lo;
        }
    }
    // the columns of A -> LDS, one row each; by_run: in the order in which a lane's sums of a product are 16 neighbouring columns
    static __device__ __forceinline__ void stage_a(const MergeArgs& g, bf16_t* sh_a, int k0, int lane, int wave, bool by_run) {
        const bool f32 = g.lora_f32 != 0;
        constexpr int NI = (RP / 4 + 7) / 8;          // items of a wave: 64 columns times eight ranks
        uint32_t a[NI > 0 ? NI : 1][8];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int item = 8 * i + wave, j0 = (item >> 1) * 8, kk = k0 + (item & 1) * 64 + lane;
            const uint32_t off = (uint32_t)(kk < g.K ? kk : g.K - 1);
            if (item < RP / 4) {
                auto load = [&](auto T_) {
                    typedef decltype(T_) T;
#pragma unroll
                    for (int e = 0; e < 8; ++e) a[i][e] = ((const T*)g.A + (int64_t)(j0 + e < g.r ? j0 + e : g.r - 1) * g.K)[off];
                };
                if (f32) load(uint32_t{});
                else load(uint16_t{});
            }
        }
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int item = 8 * i + wave, j0 = (item >> 1) * 8;
            if (item < RP / 4) {
                u32x4 hi, lo;
                merge_split8(g, a[i], false, 1.0f, j0, hi, lo);
                const int at = by_run ? (lane & 32) + (lane & 3) + 2 * (lane & 12) + ((lane & 16) >> 2) : lane;
                bf16_t* to = sh_a + ((item & 1) * 64 + at) * FP + j0;
                *(u32x4*)to = hi;
                *(u32x4*)(to + MG_T * FP) = lo;
            }
        }
    }
    // the update, transposed: acc[j][q] is row wq*32 + (lane & 31), LDS row wh*64 + j*32 + 8*(q >> 2) + 4*(lane >> 5) + (q & 3) of sh_a
    static __device__ __forceinline__ void product(f32x16 (&acc)[2], const bf16_t* sh_a, const bf16_t* sh_b, int lane, int wq, int wh) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[j][q] = 0.0f;
        const bf16_t* pa = sh_a + (wh * 64 + (lane & 31)) * FP + (lane >> 5) * 8;
        const bf16_t* pb = sh_b + (wq * 32 + (lane & 31)) * FP + (lane >> 5) * 8;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const bf16x8 bh = *(const bf16x8*)(pb + ks * 16), bl = *(const bf16x8*)(pb + MG_T * FP + ks * 16);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const bf16x8 ah = *(const bf16x8*)(pa + j * 32 * FP + ks * 16), al = *(const bf16x8*)(pa + (MG_T + j * 32) * FP + ks * 16);
                acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bl, acc[j], 0, 0, 0);
                acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, bh, acc[j], 0, 0, 0);
                acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bh, acc[j], 0, 0, 0);
            }
        }
    }
};

// Dynamic LDS of a block (merge_kernel's LDS)
template <int FMT, int RP, int MODE>
constexpr int mg_lds_bytes() {
    constexpr bool rounded = MODE == 0 || MODE >= 3 || FMT != XQ_FMT_FP8;
    constexpr int f = 2 * MG_T * (RP + 8) * 2, d = rounded ? MG_T * (MG_T + 8) * 2 : 64 * (MG_T + 4) * 4;
    return RP == 0 ? 16 : 2 * f + d <= 78 * 1024 ? 2 * f + d : f + (f > d ? f : d);
}

// N values are rounded to bf16 and come back as floats: pairs[i] the packed results
template <int N>
__device__ __forceinline__ void round_pairs(const float* v, uint32_t* pairs, float* out) {
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
        pairs[i] = pack_bf16x2(v[2 * i], v[2 * i + 1]);
        out[2 * i] = __uint_as_float(pairs[i] << 16);
        out[2 * i + 1] = __uint_as_float(pairs[i] & 0xffff0000u);
    }
}

// 16 consecutive 4-bit codes of one scale -> fp32 values, by pairs: the values of val4 (xq_common.h).  int4: a byte 0x0n read as
// e4m3 is n * 2^-9, and n - 8 is exact.
template <int FMT>
__device__ __forceinline__ void values16(float (&v)[16], uint32_t w0, uint32_t w1, float s, const float* levels) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const uint32_t w = u ? w1 : w0;
        float* o = v + 8 * u;
        if constexpr (FMT == XQ_FMT_INT4) {
            const uint32_t ev = w & 0x0f0f0f0fu, od = (w >> 4) & 0x0f0f0f0fu;
            const f32x2 e01 = e4m3x2_to_f32(ev, false), e23 = e4m3x2_to_f32(ev, true);
            const f32x2 o01 = e4m3x2_to_f32(od, false), o23 = e4m3x2_to_f32(od, true);
            const float n[8] = {e01[0], o01[0], e01[1], o01[1], e23[0], o23[0], e23[1], o23[1]};
#pragma unroll
            for (int i = 0; i < 8; ++i) o[i] = __builtin_fmaf(n[i], 512.0f, -8.0f) * s;
        } else if constexpr (FMT == XQ_FMT_NVFP4) {
            const f32x2 x0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 0), x1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 1);
            const f32x2 x2 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 2), x3 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 3);
            o[0] = x0[0] * s; o[1] = x0[1] * s; o[2] = x1[0] * s; o[3] = x1[1] * s;
            o[4] = x2[0] * s; o[5] = x2[1] * s; o[6] = x3[0] * s; o[7] = x3[1] * s;
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) o[i] = levels[(w >> (4 * i)) & 0xfu] * s;
        }
    }
}

// MODE: MergeArgs::mode, a template argument because the passes below are bound by their vector instructions: tested at run time,
// element by element, it left 64 small blocks with a branch each in the middle of the pass.
// Measured on [12288, 4096], r 32, us: with one tile a block and panels of split factors prepared by a launch before it, block-fp8
// publish 36.2, int4 41.2 (requantise 50.1), nvfp4 41.4 (absmax and codes 102.4), nf4 43.6 (53.7); as it stands 33.3, 38.0 (49.7),
// 37.9 (88.3), 38.9 (52.5).  The same sums read as 32-column pieces of 32 rows, straight from the product's registers without the
// trip through LDS, took 41 to 66: rows of 32 bytes keep the address units busy, and the runs do not fit the registers.
template <int FMT, int RP, int MODE>
__global__ void __launch_bounds__(512, 4) merge_kernel(MergeArgs g) {
    constexpr bool FP8 = FMT == XQ_FMT_FP8;
    constexpr bool ROUNDED = MODE == 0 || MODE >= 3 || !FP8;            // sums of bf16 values (4-bit decoders return bf16)
    // the update's tile in LDS between its product and the row-contiguous pass: bf16 where it is rounded to that anyway, all of
    // it at once, otherwise fp32 by halves of 64 rows
    constexpr int DP = ROUNDED ? MG_T + 8 : MG_T + 4; // its row pitch (elements)
    constexpr int DN = ROUNDED ? 1 : 2;
    constexpr int D_BYTES = RP == 0 ? 0 : ROUNDED ? MG_T * DP * 2 : 64 * DP * 4;
    asm volatile("" ::"s"(g.packed), "s"(g.scales), "s"(g.global_scale), "s"(g.group), "s"(g.scale_dtype), "s"(g.N), "s"(g.K),
                 "s"(g.A), "s"(g.B), "s"(g.lora_f32), "s"(g.r), "s"(g.scaling), "s"(g.out), "s"(g.packed_out), "s"(g.scales_out));
    // (all arguments in scalar registers after one round trip)
    typedef MergeFactors<RP> F;
    constexpr int F_BYTES = F::BYTES;
    constexpr bool APART = 2 * F_BYTES + D_BYTES <= 78 * 1024;       // B's tile beside the update's; otherwise in its place
    constexpr int LDS = RP == 0 ? 16 : APART ? 2 * F_BYTES + D_BYTES : F_BYTES + (F_BYTES > D_BYTES ? F_BYTES : D_BYTES);
    extern __shared__ __attribute__((aligned(16))) uint8_t mg_lds[];
    static_assert(LDS == mg_lds_bytes<FMT, RP, MODE>());
    bf16_t* const sh_a = (bf16_t*)mg_lds;
    bf16_t* const sh_b = (bf16_t*)(mg_lds + F_BYTES);
    uint8_t* const sh_d = mg_lds + (APART ? 2 * F_BYTES : F_BYTES);
    __shared__ float sh_amax[2][8];
    __shared__ float sh_level[FMT == XQ_FMT_NF4 ? 16 : 1];
    __shared__ Nf4Bucket sh_bucket[MODE == 5 ? 32 : 1];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wq = wave & 3, wh = wave >> 2;          // the product: rows wq*32 .. +31, columns wh*64 .. +63
    const int rrow = tid >> 3, rcol = (tid & 7) * 16; // the pass: a run of 16 columns of the rows rrow and 64 + rrow
    if constexpr (FMT == XQ_FMT_NF4) {
        if (tid < 16) sh_level[tid] = kNf4Level[tid];
        if constexpr (MODE == 5)
            if (tid >= 64 && tid < 96) sh_bucket[tid - 64] = nf4_bucket(tid - 64);
        lds_barrier();
    }

    const uint32_t tiles_n = (uint32_t)((g.N + MG_T - 1) / MG_T), tiles_k = (uint32_t)((g.K + MG_T - 1) / MG_T);
    int kt, nt;
    int64_t first, last;
    merge_tiles(g.run, tiles_n, tiles_k, first, last, nt, kt);

    const bool run_scale = !FP8 && (g.group & 15) == 0;
    const float gs = FMT == XQ_FMT_NVFP4 ? g.global_scale[0] : 1.0f;

    F factors;
    // the codes and scales of this lane's runs.  Indices past the end are clamped and their results dropped
    u32x4 wr[2];                                      // fp8: 16 bytes; 4-bit: 8 bytes (first two words)
    uint32_t sraw[2];                                 // 4-bit: the run's scale (group % 16 == 0), raw
    float tscale = 1.0f;                              // fp8: the tile's
    auto load_codes = [&](int nt_, int kt_) {
        if (FP8) tscale = ((const float*)g.scales)[(int64_t)nt_ * tiles_k + kt_];
        const int k = kt_ * MG_T + rcol < g.K ? kt_ * MG_T + rcol : g.K - 16;       // K % 16 == 0
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int nr = nt_ * MG_T + h * 64 + rrow;
            const int64_t nrow = nr < g.N ? nr : g.N - 1;
            if (FP8) wr[h] = *(const u32x4*)(g.packed + nrow * g.K + k);
            else {
                const u32x2 t = *(const u32x2*)(g.packed + ((nrow * g.K + k) >> 1));
                wr[h] = u32x4{t[0], t[1], 0u, 0u};
                const int64_t si = run_scale ? (nrow * g.K + k) / g.group : 0;
                sraw[h] = g.scale_dtype == XQ_SCALE_F32 ? ((const uint32_t*)g.scales)[si]
                        : g.scale_dtype == XQ_SCALE_BF16 ? ((const uint16_t*)g.scales)[si] : g.scales[si];
            }
        }
    };
    float amax3 = 0.0f;                               // mode 3: over all of this block's tiles
    int strip = -1, parity = 0;
    if (first < last) {
        if constexpr (RP > 0) factors.load_b(g, nt * MG_T, tid, wave);
        load_codes(nt, kt);
    }
    for (int64_t t = first; t < last; ++t, parity ^= 1) {
        const int n0 = nt * MG_T, k0 = kt * MG_T, k = k0 + rcol;
        // ---- 1. the update
        f32x16 acc[2];
        if constexpr (RP > 0) {
            const bool fresh = kt != strip;
            if (t > first && (fresh || !APART)) lds_barrier();       // the tile before this one has been read
            if (fresh) {
                strip = kt;
                F::stage_a(g, sh_a, k0, lane, wave, false);
            }
            factors.store_b(g, sh_b, tid, wave);
            lds_barrier();
            F::product(acc, sh_a, sh_b, lane, wq, wh);
            if (!APART) lds_barrier();                // B's tile is dead
        }
        const u32x4 wc[2] = {wr[0], wr[1]};
        const uint32_t sc_raw[2] = {sraw[0], sraw[1]};
        const float tile_scale = tscale;
        const int kt_tile = kt, nt_tile = nt;
        if (++nt == (int)tiles_n) { nt = 0; ++kt; }
        if (t + 1 < last) {                           // the next tile's, while this one is decoded
            if constexpr (RP > 0) factors.load_b(g, nt * MG_T, tid, wave);
            load_codes(nt, kt);
        }

        // ---- 2. decode, add
        float m[MODE == 2 ? 32 : 1];
        float amax = 0.0f;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int64_t n = n0 + h * 64 + rrow;
            const bool ok = n < g.N && k < g.K;       // K % 16 == 0: runs are all in or all out
            float v[16], x[16], d[16];
            if constexpr (RP > 0) {
                if (h < DN) {
                    if (h > 0) lds_barrier();         // the first half has been read
                    if (DN == 1 || (wq >> 1) == h) {
                        const int row = (DN == 1 ? wq : wq & 1) * 32 + (lane & 31);
#pragma unroll
                        for (int j = 0; j < 2; ++j)
#pragma unroll
                            for (int q = 0; q < 16; q += 4) {
                                const int col = wh * 64 + j * 32 + 2 * q + 4 * (lane >> 5);
                                if constexpr (ROUNDED)
                                    *(u32x2*)((bf16_t*)sh_d + row * DP + col) = u32x2{pack_bf16x2(acc[j][q], acc[j][q + 1]), pack_bf16x2(acc[j][q + 2], acc[j][q + 3])};
                                else                  // (a gap of 16 bytes in mid row: the pass's reads are free of conflicts)
                                    *(f32x4*)((float*)sh_d + row * DP + col + wh * 4) = f32x4{acc[j][q], acc[j][q + 1], acc[j][q + 2], acc[j][q + 3]};
                            }
                    }
                    lds_barrier();
                }
                if constexpr (ROUNDED) {
                    const u32x4* p = (const u32x4*)((const bf16_t*)sh_d + (h * 64 + rrow) * DP + rcol);
                    const u32x4 a = p[0], b = p[1];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        d[2 * i] = __uint_as_float(a[i] << 16); d[2 * i + 1] = __uint_as_float(a[i] & 0xffff0000u);
                        d[8 + 2 * i] = __uint_as_float(b[i] << 16); d[8 + 2 * i + 1] = __uint_as_float(b[i] & 0xffff0000u);
                    }
                } else {
                    const f32x4* p = (const f32x4*)((const float*)sh_d + rrow * DP + rcol + (rcol >> 6) * 4);
#pragma unroll
                    for (int i = 0; i < 16; ++i) d[i] = p[i >> 2][i & 3];
                }
            } else {
#pragma unroll
                for (int i = 0; i < 16; ++i) d[i] = 0.0f;
            }
            if (FP8) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const f32x2 lo = e4m3x2_to_f32(wc[h][i], false), hi = e4m3x2_to_f32(wc[h][i], true);
                    v[4 * i] = lo[0] * tile_scale; v[4 * i + 1] = lo[1] * tile_scale;
                    v[4 * i + 2] = hi[0] * tile_scale; v[4 * i + 3] = hi[1] * tile_scale;
                }
            } else if (run_scale) {
                const uint32_t sr = sc_raw[h];
                const float srun = g.scale_dtype == XQ_SCALE_F32 ? __uint_as_float(sr)
                                 : g.scale_dtype == XQ_SCALE_BF16 ? __uint_as_float(sr << 16) : e4m3_to_f32((uint8_t)sr);
                values16<FMT>(v, wc[h][0], wc[h][1], FMT == XQ_FMT_NVFP4 ? srun * gs : srun, sh_level);
            } else {
                // groups that are not multiples of 16 (never with the reference's formats): per-element lookup
                const int64_t nrow = n < g.N ? n : g.N - 1;
                for (int i = 0; i < 16; ++i) {
                    const float sc = load_scale(g.scales, (nrow * g.K + (k < g.K ? k : 0) + i) / g.group, g.scale_dtype);
                    const float u = val4<FMT>((wc[h][i >> 3] >> (4 * (i & 7))) & 0xfu, FMT == XQ_FMT_NVFP4 ? sc * gs : sc);
#pragma unroll
                    for (int e = 0; e < 16; ++e) v[e] = e == i ? u : v[e];
                }
            }
            uint32_t px[8];                           // the values as bf16 pairs (ROUNDED)
            if constexpr (ROUNDED) {
                round_pairs<16>(v, px, v);
#pragma unroll
                for (int i = 0; i < 16; ++i) x[i] = v[i] + d[i];
                round_pairs<16>(x, px, x);
            } else {
#pragma unroll
                for (int i = 0; i < 16; ++i) x[i] = v[i] + d[i];
            }
            if constexpr (MODE == 2 || MODE == 3 || MODE >= 5) {
                float hm = 0.0f;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    if constexpr (MODE == 2) m[h * 16 + i] = x[i];
                    hm = fmaxf(hm, fabsf(x[i]));
                }
                amax = fmaxf(MODE >= 5 ? 0.0f : amax, ok ? hm : 0.0f);
            }
            if constexpr (MODE == 2) {
            } else if constexpr (MODE == 3) {
                amax3 = fmaxf(amax3, amax);
            } else if constexpr (MODE == 5) {
                // NF4 (ops/quantize/nf4_quantize.py:20-56): a 64-element group is the runs of four neighbouring lanes;
                // scale = max(absmax, 1e-12), code = encode(clamp(x * (1 / scale), +-1))
#pragma unroll
                for (int off = 1; off <= 2; off <<= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
                if (ok) {
                    const float sc = fmaxf(amax, 1e-12f), inv = 1.0f / sc;
                    uint32_t lo = 0, hi = 0;
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        lo |= nf4_code(__builtin_amdgcn_fmed3f(x[i] * inv, -1.0f, 1.0f), sh_bucket) << (4 * i);
                        hi |= nf4_code(__builtin_amdgcn_fmed3f(x[8 + i] * inv, -1.0f, 1.0f), sh_bucket) << (4 * i);
                    }
                    *(u32x2*)(g.codes_out + ((n * g.K + k) >> 1)) = u32x2{lo, hi};
                    if ((tid & 3) == 0) g.scales_out[(n * g.K + k) >> 6] = sc;
                }
            } else if constexpr (MODE >= 6) {
                // int4: a 128-element group is the tile's whole row, the runs of eight neighbouring lanes (K % 128 == 0)
#pragma unroll
                for (int off = 1; off <= 4; off <<= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
                if (ok) {
                    const int64_t gi = (n * g.K + k0) >> 7;
                    uint32_t pk[2] = {0u, 0u};
                    if constexpr (MODE == 6) {
                        // scale = bf16(absmax / 7); code = clamp(rne(x / scale), -7, 7) + 8, all zero codes (8) for a zero group
                        const bf16_t sb = to_bf16(amax / 7.0f);
                        const float sc = bf16_to_f32(sb);
                        if ((tid & 7) == 0) ((bf16_t*)g.scales_out)[gi] = sb;
                        if (sc > 1e-30f && sc <= 3.0e38f) {
                            // x and sc have 8 significant bits: a quotient that is no tie lies 2^-12 or more off one, far beyond
                            // the error of x * (1 / sc), and the residual step returns ties (half integers) exactly -- the rounded
                            // quotient's codes with 3 instructions for the division's 10 (an infinite scale leaves finite values
                            // at code 8: the division's case)
                            const float inv = 1.0f / sc;
#pragma unroll
                            for (int i = 0; i < 16; ++i) {
                                const float y = x[i] * inv, q = __builtin_fmaf(__builtin_fmaf(-y, sc, x[i]), inv, y);
                                pk[i >> 3] |= (uint32_t)((int)__builtin_amdgcn_fmed3f(__builtin_rintf(q), -7.0f, 7.0f) + 8) << (4 * (i & 7));
                            }
                        } else {
#pragma unroll
                            for (int i = 0; i < 16; ++i) {
                                const float q = sc > 0.0f ? __builtin_amdgcn_fmed3f(__builtin_rintf(x[i] / sc), -7.0f, 7.0f) : 0.0f;
                                pk[i >> 3] |= (uint32_t)((int)q + 8) << (4 * (i & 7));
                            }
                        }
                    } else {
                        // ops/quantize/int4_quantize.py:12-41: scale = max(absmax, 1e-12) * (2/15); code = clamp(trunc(x * (1 /
                        // scale) + 8.5), 0, 15) with the multiplication and addition rounded separately
                        const float sc = __fmul_rn(fmaxf(amax, 1e-12f), (float)(2.0 / 15.0)), inv = 1.0f / sc;
                        if ((tid & 7) == 0) g.scales_out[gi] = sc;
#pragma unroll
                        for (int i = 0; i < 16; ++i) {
                            const float q = __fadd_rn(__fmul_rn(x[i], inv), 8.5f);
                            pk[i >> 3] |= (uint32_t)__builtin_amdgcn_fmed3f(q, 0.0f, 15.0f) << (4 * (i & 7));
                        }
                    }
                    *(u32x2*)(g.codes_out + ((n * g.K + k) >> 1)) = u32x2{pk[0], pk[1]};
                }
            } else if constexpr (MODE == 4) {
                // one nvfp4 block per run (ops/quantize/nvfp4_quantize.py:25-60,102-111): codes against the raw block
                // amax, block scale = e4m3(amax / global amax * 448)
                if (ok) {
                    float bmax = 0.0f;
#pragma unroll
                    for (int i = 0; i < 16; ++i) bmax = fmaxf(bmax, fabsf(x[i]));
                    bmax = fmaxf(bmax, 1e-12f);
                    const float q4 = 6.0f / bmax * 4.0f;
                    uint32_t lo = 0, hi = 0;
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        lo |= fp4_code4(__builtin_amdgcn_fmed3f(x[i] * q4, -24.0f, 24.0f)) << (4 * i);
                        hi |= fp4_code4(__builtin_amdgcn_fmed3f(x[8 + i] * q4, -24.0f, 24.0f)) << (4 * i);
                    }
                    *(u32x2*)(g.codes_out + ((n * g.K + k) >> 1)) = u32x2{lo, hi};
                    const float gm = fmaxf(g.gamax[0], 1e-12f);
                    const float bs = __builtin_amdgcn_fmed3f(bmax / gm * 448.0f, -448.0f, 448.0f);
                    g.bscale_out[(n * g.K + k) >> 4] = (uint8_t)(__builtin_amdgcn_cvt_pk_fp8_f32(bs, 0.0f, 0u, false) & 0xffu);
                }
            } else if (ok) {
                if constexpr (MODE == 0) {
                    bf16_t* o = (bf16_t*)g.out + n * g.K + k;
                    *(u32x4*)o = u32x4{px[0], px[1], px[2], px[3]};
                    *(u32x4*)(o + 8) = u32x4{px[4], px[5], px[6], px[7]};
                } else {
                    float* o = (float*)g.out + n * g.K + k;
#pragma unroll
                    for (int i = 0; i < 16; i += 4) *(f32x4*)(o + i) = f32x4{x[i], x[i + 1], x[i + 2], x[i + 3]};
                }
            }
        }

        // ---- 3. block-fp8: the tile's
        if constexpr (MODE == 2) {
            // block absmax -> new scale -> e4m3 bytes
            amax = wave_max63(amax);
            if (lane == 63) sh_amax[parity][wave] = amax;
            lds_barrier();
            const float* sm = sh_amax[parity];
            amax = fmaxf(fmaxf(fmaxf(sm[0], sm[1]), fmaxf(sm[2], sm[3])), fmaxf(fmaxf(sm[4], sm[5]), fmaxf(sm[6], sm[7])));
            const float s = fmaxf(amax / 448.0f, 1e-12f);
            // one division per block; x * (1/s) is within 1.5 ulp of x / s, far inside an e4m3 rounding interval except
            // for quotients within that distance of a rounding boundary
            const float rs = 1.0f / s;
            if (tid == 0) g.scales_out[(int64_t)nt_tile * tiles_k + kt_tile] = s;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int64_t n = n0 + h * 64 + rrow;
                if (!(n < g.N && k < g.K)) continue;
                uint32_t pk[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float y[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) y[e] = __builtin_amdgcn_fmed3f(m[h * 16 + 4 * i + e] * rs, -448.0f, 448.0f);
                    uint32_t w = 0;
                    w = __builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], w, false);
                    w = __builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], w, true);
                    pk[i] = w;
                }
                *(u32x4*)(g.packed_out + n * g.K + k) = u32x4{pk[0], pk[1], pk[2], pk[3]};
            }
        }
    }

    if constexpr (MODE == 3) {       // absmax -> one atomic per block (values are non-negative: integer order = float order)
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) amax3 = fmaxf(amax3, __shfl_xor(amax3, off, 64));
        if (lane == 0) sh_amax[0][wave] = amax3;
        lds_barrier();
        if (tid == 0) {
            float t = 0.0f;
            for (int i = 0; i < 8; ++i) t = fmaxf(t, sh_amax[0][i]);
            atomicMax((unsigned int*)g.amax_out, __float_as_uint(t));
        }
    } else if (MODE == 4 && tid == 0 && blockIdx.x == 0) {
        // global scale = amax / 6 / 448 in the quantizer's operation order
        g.gscale_out[0] = fmaxf(g.gamax[0], 1e-12f) * (1.0f / 6.0f) / 448.0f;
    }
}

// merge_kernel's block-fp8 requantise for ranks up to 32, where the pass itself is short and its passage through LDS was what the time
// went to: here the codes go there instead of the update (1 byte for 4).  They arrive in LDS by direct loads while the tile before
// is finished, lie in 16-byte pieces at slot piece ^ (row & 7) of their row, are read by the lanes that hold the sums of the same
// 16 columns, and the new codes take their place and leave by whole rows.  [12288, 4096], us: r 8 25.9, r 32 30.1
// (merge_kernel's form 31.1 and 35.6, one tile a block after a preparing launch 26.9 and 32.6); of these 5 to 7 go before the first tile is complete, and 3.6 (r 8) to 4.2 for every one of the
// six that a block takes, at r 8 the rate of a copy (4.7 TB/s); without the product r 32 takes 3.5 less, without B's rows 3.5 less.
template <int RP>
__global__ void __launch_bounds__(512, 4) merge_fp8_kernel(MergeArgs g) {
    typedef MergeFactors<RP> F;
    constexpr int TILE = MG_T * MG_T;
    extern __shared__ __attribute__((aligned(16))) uint8_t mg_lds[];
    __shared__ float sh_amax[8];
    bf16_t* const sh_a = (bf16_t*)mg_lds;
    bf16_t* const sh_b = (bf16_t*)(mg_lds + F::BYTES);
    uint8_t* const sh_c = mg_lds + 2 * F::BYTES;      // two tiles of codes
    const uint32_t lds_c = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)mg_lds + 2 * F::BYTES;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wq = wave & 3, wh = wave >> 2, rrow = wq * 32 + (lane & 31), half = lane >> 5;
    const uint32_t tiles_n = (uint32_t)((g.N + MG_T - 1) / MG_T), tiles_k = (uint32_t)((g.K + MG_T - 1) / MG_T);
    int kt, nt;
    int64_t first, last;
    merge_tiles(g.run, tiles_n, tiles_k, first, last, nt, kt);
    float tscale = 1.0f;

    // this lane's two pieces of a tile on the way in and out: slot 2 * wave + i, lane
    const int io_row = wave * 16 + (lane >> 3), io_piece = ((lane & 7) ^ (lane >> 3)) * 16;        // (rows 8 apart: the same order)
    auto issue = [&](int nt_, int kt_, int buf) {
        tscale = ((const float*)g.scales)[(int64_t)nt_ * tiles_k + kt_];
        const uint8_t* base = g.packed + (int64_t)nt_ * MG_T * g.K + (int64_t)kt_ * MG_T;
        const int rows = g.N - nt_ * MG_T, cols = g.K - kt_ * MG_T;         // past the end: the last ones again
        const uint32_t col = (uint32_t)(io_piece < cols ? io_piece : cols - 16);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int row = io_row + 8 * i < rows ? io_row + 8 * i : rows - 1;
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                         :: "s"(__builtin_amdgcn_readfirstlane(lds_c + (uint32_t)buf * TILE + (wave * 2 + i) * 1024)),
                            "v"((uint32_t)row * (uint32_t)g.K + col), "s"(base) : "memory");
        }
    };

    F factors;
    int buf = 0;
    if (first < last) {
        factors.load_b(g, nt * MG_T, tid, wave);
        issue(nt, kt, 0);
        F::stage_a(g, sh_a, kt * MG_T, lane, wave, true);
        factors.store_b(g, sh_b, tid, wave);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    for (int64_t t = first; t < last; ++t, buf ^= 1) {
        const int n0 = nt * MG_T, k0 = kt * MG_T;
        const float tile_scale = tscale;
        const int scale_at = nt * (int)tiles_k + kt;
        lds_barrier();                                // codes and factors of this tile are there, the tile before has left
        f32x16 m[2];
        F::product(m, sh_a, sh_b, lane, wq, wh);
        const int strip = kt;
        if (++nt == (int)tiles_n) { nt = 0; ++kt; }
        const bool more = t + 1 < last;
        if (more) {
            factors.load_b(g, nt * MG_T, tid, wave);
            issue(nt, kt, buf ^ 1);
        }
        // decode, add
        float amax = 0.0f;
        uint8_t* const codes = sh_c + buf * TILE + rrow * MG_T;
        const int swz = rrow & 7;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int piece = wh * 4 + 2 * j + half;
            const u32x4 c = *(const u32x4*)(codes + ((piece ^ swz) << 4));
            float hm = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f32x2 lo = e4m3x2_to_f32(c[i], false), hi = e4m3x2_to_f32(c[i], true);
                m[j][4 * i] = lo[0] * tile_scale + m[j][4 * i]; m[j][4 * i + 1] = lo[1] * tile_scale + m[j][4 * i + 1];
                m[j][4 * i + 2] = hi[0] * tile_scale + m[j][4 * i + 2]; m[j][4 * i + 3] = hi[1] * tile_scale + m[j][4 * i + 3];
#pragma unroll
                for (int e = 0; e < 4; ++e) hm = fmaxf(hm, fabsf(m[j][4 * i + e]));
            }
            amax = fmaxf(amax, n0 + rrow < g.N && k0 + piece * 16 < g.K ? hm : 0.0f);      // K % 16 == 0
        }
        amax = wave_max63(amax);
        if (lane == 63) sh_amax[wave] = amax;
        lds_barrier();
        amax = fmaxf(fmaxf(fmaxf(sh_amax[0], sh_amax[1]), fmaxf(sh_amax[2], sh_amax[3])),
                     fmaxf(fmaxf(sh_amax[4], sh_amax[5]), fmaxf(sh_amax[6], sh_amax[7])));
        const float s = fmaxf(amax / 448.0f, 1e-12f), rs = 1.0f / s;       // (as in merge_kernel)
        if (tid == 0) g.scales_out[scale_at] = s;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            u32x4 pk;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float y[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] = __builtin_amdgcn_fmed3f(m[j][4 * i + e] * rs, -448.0f, 448.0f);
                uint32_t w = 0;
                w = __builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], w, false);
                w = __builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], w, true);
                pk[i] = w;
            }
            *(u32x4*)(codes + (((wh * 4 + 2 * j + half) ^ swz) << 4)) = pk;
        }
        if (more) {
            if (kt != strip) F::stage_a(g, sh_a, kt * MG_T, lane, wave, true);     // (its last reads lie before the barrier above)
            factors.store_b(g, sh_b, tid, wave);
        }
        // the next tile's codes are waited for before this one's are stored: the stores then need not be waited for
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const u32x4 out = *(const u32x4*)(sh_c + buf * TILE + (wave * 2 + i) * 1024 + lane * 16);
            const int64_t n = n0 + io_row + 8 * i;
            if (n < g.N && k0 + io_piece < g.K) *(u32x4*)(g.packed_out + n * g.K + k0 + io_piece) = out;
        }
    }
}

}  // namespace xq

using namespace xq;

// FLOP-free roofline figure of this path: bytes in + bytes out per launch
static double merge_bytes(const xq_weight* w, int mode) {
    const double n = (double)w->rows * w->cols;
    const double in = (double)xq_packed_bytes_per_expert(w) + (double)xq_scale_bytes_per_expert(w);
    return in + (mode == 0 ? 2.0 * n : mode == 1 ? 4.0 * n : mode == 3 ? 0.0 : in);
}

template <int FMT, int RP, int MODE>
static int launch_merge_one(const MergeArgs& g, unsigned grid, hipStream_t s, const char* who) {
    constexpr int lds = mg_lds_bytes<FMT, RP, MODE>();
    static std::atomic<bool> attr_set{false};   // per instantiation; the attribute call is idempotent: a race only repeats it
    if (!attr_set && lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)merge_kernel<FMT, RP, MODE>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) {
            xq_set_error("%s: cannot raise the dynamic LDS limit: %s", who, hipGetErrorString(e));
            return XQ_ERR_LAUNCH;
        }
        attr_set = true;
    }
    merge_kernel<FMT, RP, MODE><<<grid, 512, lds, s>>>(g);
    return XQ_OK;
}

template <int FMT, int MODE>
static int launch_merge_fmt(const MergeArgs& g, unsigned grid, hipStream_t s, const char* who) {
    switch (g.r_pad) {
        case 0: return launch_merge_one<FMT, 0, MODE>(g, grid, s, who);
        case 16: return launch_merge_one<FMT, 16, MODE>(g, grid, s, who);
        case 32: return launch_merge_one<FMT, 32, MODE>(g, grid, s, who);
        case 48: return launch_merge_one<FMT, 48, MODE>(g, grid, s, who);
        default: return launch_merge_one<FMT, 64, MODE>(g, grid, s, who);
    }
}

template <int RP>
static int launch_merge_fp8(const MergeArgs& g, unsigned grid, hipStream_t s, const char* who) {
    constexpr int lds = 2 * MergeFactors<RP>::BYTES + 2 * MG_T * MG_T;
    static std::atomic<bool> attr_set{false};
    if (!attr_set && lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)merge_fp8_kernel<RP>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) {
            xq_set_error("%s: cannot raise the dynamic LDS limit: %s", who, hipGetErrorString(e));
            return XQ_ERR_LAUNCH;
        }
        attr_set = true;
    }
    merge_fp8_kernel<RP><<<grid, 512, lds, s>>>(g);
    return XQ_OK;
}

static int64_t merge_ws_bytes(int64_t, int64_t, int) { return 256; }     // nothing is kept there: the least a caller has to give

extern "C" int64_t xq_merge_workspace_bytes(int64_t N, int64_t K, int r) { return merge_ws_bytes(N, K, r); }

struct Nvfp4Out {      // outputs of modes 3 and 4
    float* amax_out = nullptr;
    const float* gamax = nullptr;
    uint8_t* codes_out = nullptr;
    uint8_t* bscale_out = nullptr;
    float* gscale_out = nullptr;
};

static int launch_merge(const xq_weight* w, const void* A, const void* B, int lora_dtype, int r, float scaling, int mode,
                        void* out, void* packed_out, float* scales_out, void* workspace, int64_t workspace_bytes,
                        hipStream_t stream, const char* who, const Nvfp4Out& nv = Nvfp4Out()) {
    int rc = xq_validate_weight(w, who);
    if (rc) return rc;
    XQ_REQUIRE(w->num_experts == 1, "%s: takes a single matrix", who);
    XQ_REQUIRE(w->format == XQ_FMT_FP8 || w->layout == XQ_LAYOUT_FLAT, "%s: dense weights are FLAT [N, K]", who);
    XQ_REQUIRE(w->cols % 16 == 0, "%s: in_features %lld must be a multiple of 16", who, (long long)w->cols);
    XQ_REQUIRE(r >= 0 && r <= 64, "%s: LoRA rank %d out of range [0, 64]", who, r);
    XQ_REQUIRE(r == 0 || (A && B), "%s: LoRA factors are NULL", who);
    XQ_REQUIRE(lora_dtype == XQ_DT_F32 || lora_dtype == XQ_DT_BF16, "%s: bad lora_dtype", who);
    XQ_REQUIRE(xq_aligned(w->packed, 16), "%s: packed weight must be 16-byte aligned", who);
    if (w->rows == 0 || w->cols == 0) return XQ_OK;
    MergeArgs g;
    g.packed = (const uint8_t*)w->packed; g.scales = (const uint8_t*)w->scales; g.global_scale = w->global_scale;
    g.fmt = w->format; g.group = w->group; g.scale_dtype = w->scale_dtype;
    g.N = (int32_t)w->rows; g.K = (int32_t)w->cols;
    g.A = A; g.B = B; g.lora_f32 = lora_dtype == XQ_DT_F32; g.r = r; g.r_pad = r <= 0 ? 0 : ((r + 15) / 16) * 16;
    g.scaling = scaling; g.mode = mode; g.out = out; g.packed_out = (uint8_t*)packed_out; g.scales_out = scales_out;
    g.amax_out = nv.amax_out; g.gamax = nv.gamax; g.codes_out = nv.codes_out; g.bscale_out = nv.bscale_out; g.gscale_out = nv.gscale_out;
    XQ_REQUIRE(r == 0 || (workspace && xq_aligned(workspace, 256) && workspace_bytes >= merge_ws_bytes(w->rows, w->cols, r)),
               "%s: workspace missing, misaligned or smaller than xq_merge_workspace_bytes()", who);
    // Blocks of one strip each where none has more tiles that way than an equal share has: what is read and written at a time is whole
    // rows then.  [12288, 4096] r 32, us: block-fp8 31.6 -> 30.3, int4 the same; [12288, 4224] 35.6 -> 34.1, int4 57.6 -> 55.2.  Where
    // the strips do not divide the blocks that well the equal share is better: [8192, 5120] (five tiles against six) int4 43 against 48
    const int64_t tk = xq_cdiv(w->cols, MG_T), tn = xq_cdiv(w->rows, MG_T), share = xq_cdiv(tk * tn, MG_BLOCKS);
    g.run = tk * xq_cdiv(tn, share) <= MG_BLOCKS ? (int)share : 0;
    const unsigned grid = (unsigned)(g.run ? tk * xq_cdiv(tn, share) : tk * tn < MG_BLOCKS ? tk * tn : MG_BLOCKS);
    const bool timed = xq_profile_mark_begin(stream, merge_bytes(w, mode));
    rc = XQ_ERR_UNSUPPORTED;
#define XQ_MERGE(FMT, MODE) if (w->format == FMT && mode == MODE) rc = launch_merge_fmt<FMT, MODE>(g, grid, stream, who)
    if (mode == 2 && (g.r_pad == 16 || g.r_pad == 32) && g.K <= (1 << 23)) {       // (32-bit offsets in a tile)
        rc = g.r_pad == 16 ? launch_merge_fp8<16>(g, grid, stream, who) : launch_merge_fp8<32>(g, grid, stream, who);
    } else {
        XQ_MERGE(XQ_FMT_FP8, 0); XQ_MERGE(XQ_FMT_FP8, 1); XQ_MERGE(XQ_FMT_FP8, 2); XQ_MERGE(XQ_FMT_FP8, 3);
        XQ_MERGE(XQ_FMT_INT4, 0); XQ_MERGE(XQ_FMT_INT4, 1); XQ_MERGE(XQ_FMT_INT4, 3); XQ_MERGE(XQ_FMT_INT4, 6); XQ_MERGE(XQ_FMT_INT4, 7);
        XQ_MERGE(XQ_FMT_NVFP4, 0); XQ_MERGE(XQ_FMT_NVFP4, 1); XQ_MERGE(XQ_FMT_NVFP4, 3); XQ_MERGE(XQ_FMT_NVFP4, 4);
        XQ_MERGE(XQ_FMT_NF4, 0); XQ_MERGE(XQ_FMT_NF4, 1); XQ_MERGE(XQ_FMT_NF4, 3); XQ_MERGE(XQ_FMT_NF4, 5);
    }
#undef XQ_MERGE
    if (timed) xq_profile_mark_end(stream);
    if (rc) return rc;
    XQ_CHECK_LAUNCH(who);
    return XQ_OK;
}

extern "C" int xq_merge_dense(const xq_weight* w, const void* lora_A, const void* lora_B, int lora_dtype, int r,
                              float scaling, void* out, int out_dtype, void* workspace, int64_t workspace_bytes,
                              void* stream) {
    XQ_REQUIRE(out_dtype == XQ_DT_BF16 || out_dtype == XQ_DT_F32, "xq_merge_dense: bad out_dtype");
    XQ_REQUIRE(out && xq_aligned(out, 16), "xq_merge_dense: out is NULL or not 16-byte aligned");
    return launch_merge(w, lora_A, lora_B, lora_dtype, r, scaling, out_dtype == XQ_DT_BF16 ? 0 : 1, out, nullptr, nullptr,
                        workspace, workspace_bytes, (hipStream_t)stream, "xq_merge_dense");
}

extern "C" int xq_merge_requant_fp8(const xq_weight* w, const void* lora_A, const void* lora_B, int lora_dtype, int r,
                                    float scaling, void* packed_out, float* scales_out, void* workspace,
                                    int64_t workspace_bytes, void* stream) {
    XQ_REQUIRE(w && w->format == XQ_FMT_FP8, "xq_merge_requant_fp8: the weight must be block_fp8");
    XQ_REQUIRE(packed_out && scales_out && xq_aligned(packed_out, 16), "xq_merge_requant_fp8: NULL or misaligned output");
    return launch_merge(w, lora_A, lora_B, lora_dtype, r, scaling, 2, nullptr, packed_out, scales_out, workspace, workspace_bytes,
                        (hipStream_t)stream, "xq_merge_requant_fp8");
}

extern "C" int xq_merge_amax(const xq_weight* w, const void* lora_A, const void* lora_B, int lora_dtype, int r, float scaling,
                             float* amax_out, void* workspace, int64_t workspace_bytes, void* stream) {
    XQ_REQUIRE(amax_out, "xq_merge_amax: amax_out is NULL");
    int rc = launch_zero_fill(amax_out, 4, (hipStream_t)stream);
    if (rc) return rc;
    Nvfp4Out nv;
    nv.amax_out = amax_out;
    return launch_merge(w, lora_A, lora_B, lora_dtype, r, scaling, 3, nullptr, nullptr, nullptr, workspace, workspace_bytes,
                        (hipStream_t)stream, "xq_merge_amax", nv);
}

extern "C" int xq_merge_requant_nvfp4(const xq_weight* w, const void* lora_A, const void* lora_B, int lora_dtype, int r,
                                      float scaling, const float* global_amax, void* codes_out, void* block_scales_out,
                                      float* global_scale_out, void* workspace, int64_t workspace_bytes, void* stream) {
    XQ_REQUIRE(w && w->format == XQ_FMT_NVFP4 && w->group == 16, "xq_merge_requant_nvfp4: the weight must be nvfp4 with 16-element blocks");
    XQ_REQUIRE(global_amax && codes_out && block_scales_out && global_scale_out && xq_aligned(codes_out, 8),
               "xq_merge_requant_nvfp4: NULL or misaligned output");
    XQ_REQUIRE((const void*)global_scale_out != (const void*)w->global_scale,
               "xq_merge_requant_nvfp4: the new global scale may not overwrite the one the kernel decodes with");
    Nvfp4Out nv;
    nv.gamax = global_amax; nv.codes_out = (uint8_t*)codes_out; nv.bscale_out = (uint8_t*)block_scales_out; nv.gscale_out = global_scale_out;
    return launch_merge(w, lora_A, lora_B, lora_dtype, r, scaling, 4, nullptr, nullptr, nullptr, workspace, workspace_bytes,
                        (hipStream_t)stream, "xq_merge_requant_nvfp4", nv);
}

extern "C" int xq_merge_requant_int4(const xq_weight* w, const void* lora_A, const void* lora_B, int lora_dtype, int r,
                                     float scaling, int symmetric, void* codes_out, void* scales_out, void* workspace,
                                     int64_t workspace_bytes, void* stream) {
    XQ_REQUIRE(w && w->format == XQ_FMT_INT4 && w->layout == XQ_LAYOUT_FLAT && w->group == 128 && w->cols % 128 == 0,
               "xq_merge_requant_int4: the weight must be flat int4 with 128-element groups and in_features %% 128 == 0");
    XQ_REQUIRE(codes_out && scales_out && xq_aligned(codes_out, 8) && xq_aligned(scales_out, 4),
               "xq_merge_requant_int4: NULL or misaligned output");
    Nvfp4Out nv;
    nv.codes_out = (uint8_t*)codes_out;
    return launch_merge(w, lora_A, lora_B, lora_dtype, r, scaling, symmetric ? 6 : 7, nullptr, nullptr, (float*)scales_out,
                        workspace, workspace_bytes, (hipStream_t)stream, "xq_merge_requant_int4", nv);
}

extern "C" int xq_merge_requant_nf4(const xq_weight* w, const void* lora_A, const void* lora_B, int lora_dtype, int r,
                                    float scaling, void* codes_out, float* scales_out, void* workspace,
                                    int64_t workspace_bytes, void* stream) {
    XQ_REQUIRE(w && w->format == XQ_FMT_NF4 && w->group == 64 && w->scale_dtype == XQ_SCALE_F32 && w->cols % 64 == 0,
               "xq_merge_requant_nf4: the weight must be NF4 with fp32 scales per 64 elements and in_features %% 64 == 0");
    XQ_REQUIRE(codes_out && scales_out && xq_aligned(codes_out, 8), "xq_merge_requant_nf4: NULL or misaligned output");
    Nvfp4Out nv;
    nv.codes_out = (uint8_t*)codes_out;
    return launch_merge(w, lora_A, lora_B, lora_dtype, r, scaling, 5, nullptr, nullptr, scales_out, workspace, workspace_bytes,
                        (hipStream_t)stream, "xq_merge_requant_nf4", nv);
}
