// Low-rank helper kernels (see xq_lora.h).  bf16 MFMA, fp32 accumulate.
#include "xq_lora.h"
#include <atomic>

namespace xq {

// ------------------------------------------------------------------ zero fill
__global__ void __launch_bounds__(256) zero_fill_kernel(u32x4* p, int64_t n16, uint8_t* tail, int tail_bytes) {
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n16) p[i] = u32x4{0, 0, 0, 0};
    if (i == 0)
        for (int t = 0; t < tail_bytes; ++t) tail[t] = 0;
}

int launch_zero_fill(void* p, int64_t bytes, hipStream_t stream) {
    if (bytes <= 0) return XQ_OK;
    XQ_REQUIRE(xq_aligned(p, 16), "zero_fill: pointer not 16-byte aligned");
    int64_t n16 = bytes / 16;
    int tail = (int)(bytes - n16 * 16);
    int64_t blocks = xq_cdiv(n16 > 0 ? n16 : 1, 256);
    zero_fill_kernel<<<dim3((unsigned)blocks), 256, 0, stream>>>((u32x4*)p, n16, (uint8_t*)p + n16 * 16, tail);
    XQ_CHECK_LAUNCH("zero_fill");
    return XQ_OK;
}

// ------------------------------------------------------------------ factor prep
__global__ void __launch_bounds__(256) factor_prep_kernel(const void* in, int in_f32, int64_t R_in, int64_t C_in,
                                                          int transpose, bf16_t* out, int64_t R_out, int64_t C_out,
                                                          int64_t total) {
    int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= total) return;
    int64_t per = R_out * C_out;
    int64_t e = t / per, rem = t - e * per;
    int64_t i = rem / C_out, j = rem - i * C_out;
    int64_t si = transpose ? j : i, sj = transpose ? i : j;
    float v = 0.0f;
    if (si < R_in && sj < C_in) {
        int64_t idx = e * R_in * C_in + si * C_in + sj;
        v = in_f32 ? ((const float*)in)[idx] : bf16_to_f32(((const bf16_t*)in)[idx]);
    }
    out[t] = to_bf16(v);
}

int launch_factor_prep(const void* in, int in_dtype, int64_t R_in, int64_t C_in, bool transpose, bf16_t* out,
                       int64_t R_out, int64_t C_out, int64_t num_experts, hipStream_t stream) {
    int64_t total = num_experts * R_out * C_out;
    if (total == 0) return XQ_OK;
    factor_prep_kernel<<<dim3((unsigned)xq_cdiv(total, 256)), 256, 0, stream>>>(in, in_dtype == XQ_DT_F32, R_in, C_in,
                                                                                transpose, out, R_out, C_out, total);
    XQ_CHECK_LAUNCH("factor_prep");
    return XQ_OK;
}

// A block converts one tile of a destination panel through LDS -- 16 x 256 (rows x columns) of a wide panel, 256 x 16
// of a tall one -- so that both the source and the destination are touched in whole row pieces whichever way the job
// transposes: e.g. a transposing job into a wide panel reads 256 source rows of 16 entries (one contiguous run when
// the factor is 16 wide) and writes 16 destination rows of 512 bytes.  (Element by element, the transposing jobs of
// an expert bank read 4 bytes of every 64-byte row piece per instruction: 61 us for the panels of 128 experts.)
// Every load is unconditional (indices past the source clamped onto it, the value replaced by zero afterwards): with a
// branch around them the compiler waits for each load before it issues the next, sixteen round trips per tile.
constexpr int PP_S = 16, PP_L = 256;
template <bool F32>
__global__ void __launch_bounds__(256) panel_prep_kernel(PanelJobs j) {
    __shared__ float tile[PP_L][PP_S + 1];      // [index along the tile's long side][along its short side]
    const int k = blockIdx.y, tid = threadIdx.x;
    const int64_t R_in = j.R_in[k], C_in = j.C_in[k], C_out = j.C_out[k], R_out = j.R_out[k], pitch = j.pitch[k];
    const bool tr = j.transpose[k] != 0, shared = j.n_src[k] == 1;
    const void* in = j.in[k];
    bf16_t* out = j.out[k];
    const int64_t e_stride = j.e_stride[k];
    const bool wide = C_out >= R_out;           // the long side runs along the destination's columns
    const int64_t TRW = wide ? PP_S : PP_L, TCW = wide ? PP_L : PP_S;
    const int64_t tiles_r = (R_out + TRW - 1) / TRW, tiles_c = (C_out + TCW - 1) / TCW;
    const int64_t total = tiles_r * tiles_c * j.n_out[k];
    const bool load_long_first = wide != tr;    // consecutive threads walk along the source's rows
    for (int64_t t = blockIdx.x; t < total; t += gridDim.x) {
        const int64_t e = t / (tiles_r * tiles_c), rem = t - e * (tiles_r * tiles_c);
        const int64_t i0 = (rem / tiles_c) * TRW, c0 = (rem % tiles_c) * TCW;
        const int64_t base = (shared ? 0 : e) * R_in * C_in;
        float val[PP_S];
        uint32_t keep = 0xffffu;
#pragma unroll
        for (int u = 0; u < PP_S; ++u) {
            const int idx = u * 256 + tid;
            const int l = load_long_first ? idx % PP_L : idx / PP_S, sh = load_long_first ? idx / PP_L : idx % PP_S;
            const int64_t i = i0 + (wide ? sh : l), c = c0 + (wide ? l : sh);
            const int64_t si = tr ? c : i, sj = tr ? i : c;
            const int64_t src = base + (si < R_in ? si : R_in - 1) * C_in + (sj < C_in ? sj : C_in - 1);
            val[u] = F32 ? ((const float*)in)[src] : bf16_to_f32(((const bf16_t*)in)[src]);
            if (!(si < R_in && sj < C_in)) keep &= ~(1u << u);
        }
#pragma unroll
        for (int u = 0; u < PP_S; ++u) {
            const int idx = u * 256 + tid;
            const int l = load_long_first ? idx % PP_L : idx / PP_S, sh = load_long_first ? idx / PP_L : idx % PP_S;
            tile[l][sh] = (keep >> u) & 1u ? val[u] : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < PP_S; ++u) {
            const int idx = u * 256 + tid;      // consecutive threads walk along the destination's rows
            const int l = wide ? idx % PP_L : idx / PP_S, sh = wide ? idx / PP_L : idx % PP_S;
            const int64_t i = i0 + (wide ? sh : l), c = c0 + (wide ? l : sh);
            if (i < R_out && c < C_out) out[e * e_stride + i * pitch + c] = to_bf16(tile[l][sh]);
        }
        __syncthreads();
    }
}

// The same where four elements of a source row and of a destination row are one aligned piece (panel_vec): 16-byte loads of fp32
// factors, 8-byte stores, and no LDS where nothing is transposed.  By single elements the kernel is bound by address arithmetic and
// 2-byte stores, at half the rate of a copy.  Panels of 128 experts (hidden 2048, intermediate 768, r 16; 69 MB read, 35 written): 33 us by elements, 23 here;
// 64 experts with factors shared by all on one side 15 and 8.
template <bool F32>
__global__ void __launch_bounds__(256) panel_prep_vec_kernel(PanelJobs j) {
    __shared__ float tile[PP_L][PP_S + 1];
    const int k = blockIdx.y, tid = threadIdx.x;
    const int R_in = (int)j.R_in[k], C_in = (int)j.C_in[k], C_out = (int)j.C_out[k], R_out = (int)j.R_out[k];
    const bool tr = j.transpose[k] != 0, wide = C_out >= R_out;
    const int TRW = wide ? PP_S : PP_L, TCW = wide ? PP_L : PP_S;
    const uint32_t tiles_c = (uint32_t)(C_out + TCW - 1) / TCW, per = (uint32_t)(R_out + TRW - 1) / TRW * tiles_c;
    const uint32_t total = per * (uint32_t)j.n_out[k];
    const bool load_long_first = wide != tr;
    for (uint32_t t = blockIdx.x; t < total; t += gridDim.x) {
        const uint32_t e = t / per, rem = t - e * per;
        const int i0 = (int)(rem / tiles_c) * TRW, c0 = (int)(rem % tiles_c) * TCW;
        const int64_t base = j.n_src[k] == 1 ? 0 : (int64_t)e * R_in * C_in;
        bf16_t* out = j.out[k] + e * j.e_stride[k];
        u32x4 val[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {            // (unconditional: a piece past the source is clamped onto it and dropped)
            const int idx = u * 256 + tid;
            const int l = load_long_first ? idx % 64 * 4 : idx / 4, sh = load_long_first ? idx / 64 : idx % 4 * 4;
            const int i = i0 + (wide ? sh : l), c = c0 + (wide ? l : sh);
            const int si = tr ? c : i, sj = tr ? i : c;
            const int64_t src = base + (int64_t)min(si, R_in - 1) * C_in + min(sj, C_in - 4);
            if (F32) {
                val[u] = *(const u32x4*)((const float*)j.in[k] + src);
            } else {
                const u32x2 h = *(const u32x2*)((const bf16_t*)j.in[k] + src);
                val[u] = u32x4{h[0] << 16, h[0] & 0xffff0000u, h[1] << 16, h[1] & 0xffff0000u};
            }
            const uint32_t keep = si < R_in && sj < C_in ? 0xffffffffu : 0u;
            val[u] = u32x4{val[u][0] & keep, val[u][1] & keep, val[u][2] & keep, val[u][3] & keep};
        }
        auto put = [&](int l, int sh, float v0, float v1, float v2, float v3) {
            const int i = i0 + (wide ? sh : l), c = c0 + (wide ? l : sh);
            if (i < R_out && c < C_out) *(u32x2*)(out + (int64_t)i * j.pitch[k] + c) = u32x2{pack_bf16x2(v0, v1), pack_bf16x2(v2, v3)};
        };
        if (!tr) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int idx = u * 256 + tid;
                put(wide ? idx % 64 * 4 : idx / 4, wide ? idx / 64 : idx % 4 * 4, __uint_as_float(val[u][0]), __uint_as_float(val[u][1]),
                    __uint_as_float(val[u][2]), __uint_as_float(val[u][3]));
            }
            continue;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int idx = u * 256 + tid;
            const int l = load_long_first ? idx % 64 * 4 : idx / 4, sh = load_long_first ? idx / 64 : idx % 4 * 4;
#pragma unroll
            for (int q = 0; q < 4; ++q) tile[load_long_first ? l + q : l][load_long_first ? sh : sh + q] = __uint_as_float(val[u][q]);
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int idx = u * 256 + tid;
            const int l = wide ? idx % 64 * 4 : idx / 4, sh = wide ? idx / 64 : idx % 4 * 4;
            if (wide) put(l, sh, tile[l][sh], tile[l + 1][sh], tile[l + 2][sh], tile[l + 3][sh]);
            else put(l, sh, tile[l][sh], tile[l][sh + 1], tile[l][sh + 2], tile[l][sh + 3]);
        }
        __syncthreads();
    }
}

static bool panel_vec(const PanelJobs& j) {
    for (int k = 0; k < j.n; ++k) {
        const int64_t tiles = xq_cdiv(j.R_out[k], PP_S) * xq_cdiv(j.C_out[k], PP_S) * j.n_out[k];
        if (j.C_in[k] % 4 || j.C_out[k] % 4 || j.pitch[k] % 4 || j.e_stride[k] % 4 || j.R_in[k] < 1 || j.C_in[k] < 4 || tiles >= (1ll << 31) ||
            j.R_in[k] >= (1ll << 30) || j.C_in[k] >= (1ll << 30) || j.R_out[k] >= (1ll << 30) || j.C_out[k] >= (1ll << 30) ||
            !xq_aligned(j.in[k], j.in_f32 ? 16 : 8) || !xq_aligned(j.out[k], 8))
            return false;
    }
    return true;
}

int launch_panel_prep(const PanelJobs& j, hipStream_t stream) {
    int64_t most = 0;
    for (int k = 0; k < j.n; ++k) {
        const bool wide = j.C_out[k] >= j.R_out[k];
        const int64_t t = xq_cdiv(j.R_out[k], wide ? PP_S : PP_L) * xq_cdiv(j.C_out[k], wide ? PP_L : PP_S) * j.n_out[k];
        most = t > most ? t : most;
    }
    if (j.n == 0 || most == 0) return XQ_OK;
    if (most > 16384) most = 16384;
    if (panel_vec(j)) {
        if (j.in_f32) panel_prep_vec_kernel<true><<<dim3((unsigned)most, (unsigned)j.n), 256, 0, stream>>>(j);
        else panel_prep_vec_kernel<false><<<dim3((unsigned)most, (unsigned)j.n), 256, 0, stream>>>(j);
        XQ_CHECK_LAUNCH("panel_prep");
        return XQ_OK;
    }
    if (j.in_f32) panel_prep_kernel<true><<<dim3((unsigned)most, (unsigned)j.n), 256, 0, stream>>>(j);
    else panel_prep_kernel<false><<<dim3((unsigned)most, (unsigned)j.n), 256, 0, stream>>>(j);
    XQ_CHECK_LAUNCH("panel_prep");
    return XQ_OK;
}

// ------------------------------------------------------------------ small_nt
struct SmallNtArgs {
    const bf16_t* In;
    int64_t ld_in;
    int64_t n_rows;
    int64_t Kc;
    const bf16_t* F;
    int64_t f_stride;  // elements per expert (0 = shared)
    int r_pad;
    float scale;
    bf16_t* T;
    int64_t ld_t;      // row pitch of T (and T2) in elements
    bf16_t* T2;        // optional: result columns from `split` on go to T2 (as its columns 0 ..) instead of T
    int split;
    const int32_t* offsets;
    const int32_t* tile_offsets;
    int32_t num_experts;
    // grouped, optional: row i of the product is made from row row_map[i] of In (rows gathered from a compact matrix),
    // and the gathered rows are also written to copy_out (row pitch ld_copy) -- the row permutation of a routed
    // problem rides on the pass that reads the rows first instead of being a pass of its own
    const int32_t* row_map;
    bf16_t* copy_out;
    int64_t ld_copy;
};

// 128 rows of one expert per block, a wave per 32 rows.  FJ = rows of F in use / 4 (4, 8, 12 or 16).
// Both operands are fetched with coalesced 16-byte loads (16 lanes per 256-byte row piece, 4 rows
// per instruction) and reach the MFMA operand layout through wave-private LDS tiles of 128 k per
// row (row pitch 272 B: the 16 lanes of a b128 read phase hit distinct banks); per-lane row-strided
// loads would touch 64 cache lines per instruction and leave the kernel address-unit bound.
// A wave keeps two 128-k chunks of its activation rows in flight (the factor chunk, which comes from L2, one):
// every load is unconditional -- rows past the segment and columns past the wave's K range are clamped onto
// valid ones and their values never used -- so the waits count exactly and the loads of chunk k+2 stay in
// flight while chunk k is multiplied.
// NARROW: 32 rows per block and the contraction split over its waves (eight, four beyond rank 32), whose sums meet in LDS in wave
// order.  With few rows the wide form is a fraction of the chip's waves, each a chain of Kc / 128 trips to memory (narrow_nt has both
// forms' times).
constexpr int SN_P = 136;   // LDS row pitch in bf16 elements
constexpr int sn_waves(int FJ, bool narrow) { return narrow && FJ <= 8 ? 8 : 4; }
template <int FJ, bool GATHER, bool NARROW>
__global__ void __launch_bounds__(64 * sn_waves(FJ, NARROW)) small_nt_kernel(SmallNtArgs g) {
    constexpr int NT = (FJ + 7) / 8, NW = sn_waves(FJ, NARROW);
    constexpr int TR = 128;
    constexpr int WTILE = (32 + NT * 32) * SN_P;   // bf16 elements per wave: In tile + F tile
    extern __shared__ __attribute__((aligned(16))) bf16_t sn_lds[];
    __shared__ int sh_info[3];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int rg = NARROW ? (int)(blockIdx.x / (gridDim.x >> 2)) : wave;

    int e = 0;
    int64_t row0, row_end;
    {
        // the expert whose tile range holds this block's tile: one look per thread, all loads in flight together
        // (a binary search by one thread is a chain of dependent memory round trips)
        if (tid == 0) sh_info[0] = -1;
        __syncthreads();
        const int t = NARROW ? blockIdx.x % (gridDim.x >> 2) : blockIdx.x;     // (a tile's four parts a stretch apart: experts of few rows fill only the first)
        for (int x = tid; x < g.num_experts; x += blockDim.x) {
            const int lo = g.tile_offsets[x], hi = g.tile_offsets[x + 1];
            const int o0 = g.offsets[x], o1 = g.offsets[x + 1];
            if (lo <= t && t < hi) {
                sh_info[0] = x;
                sh_info[1] = o0 + (t - lo) * TR;
                sh_info[2] = o1;
            }
        }
        __syncthreads();
        e = sh_info[0];
        if (e < 0) return;
        row0 = sh_info[1];
        row_end = sh_info[2];
        if (NARROW && row0 + rg * 32 >= row_end) return;
    }
    const bf16_t* F = g.F + (int64_t)e * g.f_stride;
    bf16_t* xs = sn_lds + wave * WTILE;          // [32][SN_P]
    bf16_t* fs = xs + 32 * SN_P;                 // [NT*32][SN_P]
    const int fr = lane & 31, fk = (lane >> 5) * 8;
    const int crow = lane >> 4, cpiece = (lane & 15) * 8;   // coalesced fetch: row within a group of 4, k offset
    const int64_t wrow0 = row0 + rg * 32;
    const int frows = g.r_pad;                   // rows of F in use (= 4 * FJ)

    f32x16 acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[n][q] = 0.0f;

    const int64_t units = (g.Kc + 127) >> 7;
    const int64_t kbeg = NARROW ? units * wave / NW << 7 : 0, kto = NARROW ? units * (wave + 1) / NW << 7 : g.Kc, kend = kto < g.Kc ? kto : g.Kc;
    const bf16_t* xp[8];
    int32_t orow[GATHER ? 8 : 1];                // GATHER: the rows of copy_out this lane's pieces belong to
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        int64_t r = wrow0 + j * 4 + crow;
        r = r < row_end ? r : row_end - 1;       // wrow0 may lie past a short segment's end: still a valid row
        r = r < 0 ? 0 : r;
        if constexpr (GATHER) {
            orow[j] = (int32_t)r;
            xp[j] = g.In + (int64_t)g.row_map[r] * g.ld_in;
        } else {
            xp[j] = g.In + r * g.ld_in;
        }
    }
    u32x4 xr[2][8], fq[FJ];
    auto fetch_x = [&](u32x4* dst, int64_t k) {  // chunk [k, k+128); pieces past kend come from the range's last piece
        int64_t kc = k + cpiece;
        kc = kc < kend ? kc : kend - 8;
#pragma unroll
        for (int j = 0; j < 8; ++j) dst[j] = *(const u32x4*)(xp[j] + kc);
    };
    auto fetch_f = [&](int64_t k) {
        int64_t kc = k + cpiece;
        kc = kc < kend ? kc : kend - 8;
#pragma unroll
        for (int j = 0; j < FJ; ++j) fq[j] = *(const u32x4*)(F + (int64_t)(j * 4 + crow) * g.Kc + kc);
    };
    auto chunk = [&](u32x4* cur, int64_t k) {    // multiply chunk k out of `cur`; refill it with chunk k + 256
        // LDS operations of one wave execute in order: the previous chunk's fragment reads are ahead of these writes
#pragma unroll
        for (int j = 0; j < 8; ++j) *(u32x4*)(xs + (j * 4 + crow) * SN_P + cpiece) = cur[j];
#pragma unroll
        for (int j = 0; j < FJ; ++j) *(u32x4*)(fs + (j * 4 + crow) * SN_P + cpiece) = fq[j];
        if constexpr (GATHER) {
            // (rows and pieces that were clamped onto valid ones are written again with the same bytes)
            int64_t kc = k + cpiece;
            kc = kc < kend ? kc : kend - 8;
            if (g.copy_out && k < kend) {
#pragma unroll
                for (int j = 0; j < 8; ++j) *(u32x4*)(g.copy_out + (int64_t)orow[j] * g.ld_copy + kc) = cur[j];
            }
        }
        fetch_f(k + 128);
        fetch_x(cur, k + 256);
        const int64_t left = kend - k;           // <= 0 for the idle second half of the last pair
        const int nsteps = (int)((left < 128 ? (left < 0 ? 0 : left) : 128) >> 4);
#pragma unroll
        for (int st = 0; st < 8; ++st) {
            if (st < nsteps) {                   // uniform
                const bf16x8 a = *(const bf16x8*)(xs + fr * SN_P + st * 16 + fk);
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
                    const bf16x8 b = (n * 32 + fr < frows) ? *(const bf16x8*)(fs + (n * 32 + fr) * SN_P + st * 16 + fk) : zero8;
                    acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[n], 0, 0, 0);
                }
            }
        }
    };
    if (!NARROW || kbeg < kend) {                // (fewer units than waves: nothing to fetch)
        fetch_x(xr[0], kbeg);
        fetch_f(kbeg);
        fetch_x(xr[1], kbeg + 128);
        for (int64_t k = kbeg; k < kend; k += 256) {
            chunk(xr[0], k);
            chunk(xr[1], k + 128);
        }
    }
    if constexpr (NARROW) {
        float* red = (float*)sn_lds;             // [NW - 1][NT][16][64] floats, over the (now dead) tiles
        __syncthreads();
        if (wave > 0) {
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int q = 0; q < 16; ++q) red[(((wave - 1) * NT + n) * 16 + q) * 64 + lane] = acc[n][q];
        }
        __syncthreads();
        if (wave > 0) return;
#pragma unroll
        for (int w = 1; w < NW; ++w)
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int q = 0; q < 16; ++q) acc[n][q] += red[(((w - 1) * NT + n) * 16 + q) * 64 + lane];
    }

    const int rgrp = (lane >> 5) * 4;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        int j = n * 32 + fr;
        if (j >= g.r_pad) continue;
        bf16_t* dst = g.T;
        int jj = j;
        if (g.T2 && j >= g.split) { dst = g.T2; jj = j - g.split; }
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            int64_t row = row0 + rg * 32 + (q & 3) + rgrp + 8 * (q >> 2);
            if (row < row_end) dst[row * g.ld_t + jj] = to_bf16(acc[n][q] * g.scale);
        }
    }
}

template <int FJ, bool GATHER, bool NARROW>
static int launch_small_nt_one(const SmallNtArgs& g, unsigned blocks, hipStream_t stream) {
    constexpr int NT = (FJ + 7) / 8, NW = sn_waves(FJ, NARROW);
    constexpr size_t lds = (size_t)NW * (32 + NT * 32) * SN_P * 2;
    static std::atomic<bool> attr_set{false};   // the attribute call is idempotent: a race only repeats it
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute((const void*)small_nt_kernel<FJ, GATHER, NARROW>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) {
            xq_set_error("small_nt: cannot raise the dynamic LDS limit: %s", hipGetErrorString(e));
            return XQ_ERR_LAUNCH;
        }
        attr_set = true;
    }
    small_nt_kernel<FJ, GATHER, NARROW><<<dim3(NARROW ? 4 * blocks : blocks), 64 * NW, lds, stream>>>(g);
    return XQ_OK;
}

template <bool GATHER, bool NARROW>
static int launch_small_nt_rows(const SmallNtArgs& g, unsigned blocks, hipStream_t stream) {
    switch (g.r_pad) {
        case 16: return launch_small_nt_one<4, GATHER, NARROW>(g, blocks, stream);
        case 32: return launch_small_nt_one<8, GATHER, NARROW>(g, blocks, stream);
        case 48: return launch_small_nt_one<12, GATHER, NARROW>(g, blocks, stream);
        default: return launch_small_nt_one<16, GATHER, NARROW>(g, blocks, stream);
    }
}

// Routed rows in blocks of 32 whose waves split the contraction, or in blocks of 128 whose waves split the rows: the first where it
// leaves a block per compute unit or less (experts' last blocks are half empty on average).  us, wide -> narrow: K 2048, two factors
// of rank 16, 1800 rows of 64 experts 18.9 -> 11.2, 6000 19.2 -> 19.7, 12000 19.5 -> 22.6; K 4096, rank 32, 16 experts: 1200 rows 48.5 ->
// 19.9 (two factors) and 31.2 -> 14.3 (one), 6000 49.6 -> 22.2 and 32.3 -> 16.5, 16000 51.5 -> 60.3.
static bool narrow_nt(int64_t n_rows, int num_experts) { return xq_cdiv(n_rows, 32) + num_experts / 2 <= num_cus(); }

int launch_small_nt(const bf16_t* In, int64_t ld_in, int64_t n_rows, int64_t Kc, const bf16_t* F, int r_pad,
                    float scale, bf16_t* T, const int32_t* offsets, const int32_t* tile_offsets,
                    int32_t num_experts, bool shared_f, hipStream_t stream, int64_t ld_t, bf16_t* T2, int split,
                    const int32_t* row_map, bf16_t* copy_out, int64_t ld_copy) {
    if (ld_t <= 0) ld_t = r_pad;
    if (T2) XQ_REQUIRE(split > 0 && split < r_pad && ld_t >= split && ld_t >= r_pad - split, "small_nt: bad split of the result columns");
    else XQ_REQUIRE(ld_t >= r_pad, "small_nt: output pitch %lld below r_pad %d", (long long)ld_t, r_pad);
    XQ_REQUIRE(r_pad > 0 && r_pad <= 64 && r_pad % 16 == 0, "small_nt: r_pad must be 16/32/48/64, got %d", r_pad);
    XQ_REQUIRE(Kc % 64 == 0, "small_nt: contraction length %lld must be a multiple of 64", (long long)Kc);
    XQ_REQUIRE(ld_in % 8 == 0 && xq_aligned(In, 16) && xq_aligned(F, 16), "small_nt: operands must be 16-byte aligned");
    if (n_rows == 0) return XQ_OK;
    XQ_REQUIRE(offsets && tile_offsets && num_experts >= 1, "small_nt: rows in expert order");
    XQ_REQUIRE(!row_map || !copy_out || (ld_copy % 8 == 0 && ld_copy >= Kc && xq_aligned(copy_out, 16)),
               "small_nt: a copy of gathered rows needs a 16-byte aligned copy_out");
    SmallNtArgs g{In, ld_in, n_rows, Kc, F, shared_f ? 0 : (int64_t)r_pad * Kc, r_pad, scale, T, ld_t, T2, split, offsets,
                  tile_offsets, num_experts, row_map, copy_out, ld_copy};
    const unsigned blocks = (unsigned)(xq_cdiv(n_rows, 128) + num_experts);
    const int rc = narrow_nt(n_rows, num_experts)
                       ? (row_map ? launch_small_nt_rows<true, true>(g, blocks, stream) : launch_small_nt_rows<false, true>(g, blocks, stream))
                       : (row_map ? launch_small_nt_rows<true, false>(g, blocks, stream) : launch_small_nt_rows<false, false>(g, blocks, stream));
    if (rc) return rc;
    XQ_CHECK_LAUNCH("small_nt");
    return XQ_OK;
}

// ------------------------------------------------------------------ dense low-rank products from the factors as they are
// 8 consecutive contraction elements of one rank of a factor, in the four forms a factor comes in; an fp32 factor is
// rounded to bf16 on its way to the MFMA.  Loads are unconditional (the caller clamps rank and position).
typedef u32x4 __attribute__((aligned(2))) u32x4_a2;
typedef u32x4 __attribute__((aligned(4))) u32x4_a4;
typedef f32x4 __attribute__((aligned(4))) f32x4_a4;
template <int MODE>
struct FactorPiece;
template <>
struct FactorPiece<kFacBf16> {
    u32x4 v;
    __device__ __forceinline__ void load(const void* F, int, int64_t Kc, int rank, int64_t k) {
        v = *(const u32x4_a2*)((const bf16_t*)F + (int64_t)rank * Kc + k);
    }
    __device__ __forceinline__ u32x4 get() const { return v; }
};
template <>
struct FactorPiece<kFacF32> {
    f32x4 a, b;
    __device__ __forceinline__ void load(const void* F, int, int64_t Kc, int rank, int64_t k) {
        const float* p = (const float*)F + (int64_t)rank * Kc + k;
        a = *(const f32x4_a4*)p;
        b = *(const f32x4_a4*)(p + 4);
    }
    __device__ __forceinline__ u32x4 get() const {
        return u32x4{pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3]), pack_bf16x2(b[0], b[1]), pack_bf16x2(b[2], b[3])};
    }
};
template <>
struct FactorPiece<kFacF32T> {
    float v[8];
    __device__ __forceinline__ void load(const void* F, int r, int64_t, int rank, int64_t k) {
        const float* p = (const float*)F + k * r + rank;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = p[(int64_t)e * r];
    }
    __device__ __forceinline__ u32x4 get() const {
        return u32x4{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
    }
};
template <>
struct FactorPiece<kFacBf16T> {
    uint32_t v[8];
    __device__ __forceinline__ void load(const void* F, int r, int64_t, int rank, int64_t k) {
        const bf16_t* p = (const bf16_t*)F + k * r + rank;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = p[(int64_t)e * r];
    }
    __device__ __forceinline__ u32x4 get() const {
        return u32x4{v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16)};
    }
};

struct LowRankBatch {
    LowRankJob job[kLowRankJobs];
    int32_t first[kLowRankJobs];      // first block of a job
    int32_t n;
    int64_t n_rows;
    int32_t splits;                   // > 1 (one product): split blockIdx.y of the contraction leaves its fp32 sums to partial
    float* partial;                   // [splits][n_rows][nf * rp]
};

// T[rows, nf * rp] = bf16(scale * In . F^T), up to kLowRankJobs products in one launch.  A block owns 16 RT rows; its NW waves
// take 64 contraction elements each in turn and their sums meet in LDS in wave order.  Activations and [r, K] factors are
// fetched in whole 128-byte lines and reach the MFMA operand layout through wave-private LDS rows: taken from memory in that
// layout, 16 rows a power of two apart land in one set of the L1 and the two loads that share a line fetch it twice (512 rows,
// K 4096, r 16: 16 us against 8).  A [K, r] factor is contiguous and is read element by element.  The next unit's loads are in
// flight while one is multiplied.  Few rows leave most of the chip idle whatever a block does, so it is made short instead:
// sixteen waves (eight for wide factors) pull a block's rows at the rate of one compute unit.  NT: column tiles of 16 ranks.
constexpr int LR_P = 72;              // LDS row pitch in bf16 elements: the 16 rows of a 16-byte fragment read fall on 16 bank quads
template <int MODE, int NT, int RT, int NW>
struct LowRankLds {
    static constexpr bool STAGE_F = MODE == kFacF32 || MODE == kFacBf16;
    static constexpr int WAVE = (RT + (STAGE_F ? NT : 0)) * 16 * LR_P;                      // bf16 elements per wave
    static constexpr size_t tiles = (size_t)NW * WAVE * 2, sums = (size_t)NW * RT * NT * 64 * 16;
    static constexpr size_t bytes = tiles > sums ? tiles : sums;
};
template <int MODE, int NT, int RT, int NW>
__global__ void __launch_bounds__(64 * NW, NW / 4) lowrank_kernel(LowRankBatch b) {
    using L = LowRankLds<MODE, NT, RT, NW>;
    extern __shared__ __attribute__((aligned(16))) unsigned char lr_lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lg = lane >> 4;
    int ji = 0;
#pragma unroll
    for (int i = 1; i < kLowRankJobs; ++i)
        if (i < b.n && (int)blockIdx.x >= b.first[i]) ji = i;
    const LowRankJob& g = b.job[ji];
    const int64_t row0 = (int64_t)((int)blockIdx.x - b.first[ji]) * (16 * RT);
    const int rp = g.rp, cols = g.nf * rp;
    bf16_t* xs = (bf16_t*)lr_lds + wave * L::WAVE;      // [16 RT][LR_P]
    bf16_t* fs = xs + RT * 16 * LR_P;                   // [16 NT][LR_P]
    // activations: 8 rows of 128 bytes per load instruction
    const bf16_t* xp[2 * RT];
#pragma unroll
    for (int i = 0; i < 2 * RT; ++i) {
        const int64_t r = row0 + i * 8 + (lane >> 3);
        xp[i] = g.In + (r < b.n_rows ? r : b.n_rows - 1) * g.ld_in + (lane & 7) * 8;
    }
    // staged factor: fp32, 4 ranks of 256 bytes per instruction; bf16, 8 ranks of 128 bytes
    constexpr int FI = MODE == kFacF32 ? 4 : 2;         // instructions per 16 ranks
    struct Unit {
        u32x4 x[2 * RT];
        u32x4 fv[L::STAGE_F ? NT * FI : 1];
        FactorPiece<L::STAGE_F ? kFacBf16 : MODE> fd[L::STAGE_F ? 1 : NT][2];
    };
    const void* fp[NT];
    int j0[NT];                                         // first rank of the tile within its factor
    bool in_job[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int f = t * 16 >= rp && g.nf > 1 ? 1 : 0;
        fp[t] = f ? g.F[1] : g.F[0];
        j0[t] = t * 16 - f * rp;
        in_job[t] = t * 16 < cols;
    }
    const int r1 = g.r - 1;
    // (a staged factor's lane offsets, in bytes from the factor: 32 bits, beside a base every lane shares)
    uint32_t fo[L::STAGE_F ? NT * FI : 1];
    if constexpr (L::STAGE_F) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int i = 0; i < FI; ++i) {
                const int j = min(j0[t] + i * (16 / FI) + (MODE == kFacF32 ? lane >> 4 : lane >> 3), r1);
                fo[t * FI + i] = MODE == kFacF32 ? ((uint32_t)j * (uint32_t)g.Kc + (lane & 15) * 4) * 4 : ((uint32_t)j * (uint32_t)g.Kc + (lane & 7) * 8) * 2;
            }
    }
    f32x4 acc[RT][NT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto load = [&](Unit& u, int unit) {
        const int64_t k = (int64_t)unit * 64;
#pragma unroll
        for (int i = 0; i < 2 * RT; ++i) u.x[i] = *(const u32x4*)(xp[i] + k);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if constexpr (L::STAGE_F) {
#pragma unroll
                for (int i = 0; i < FI; ++i) {
                    const unsigned char* base = (const unsigned char*)fp[t] + k * (MODE == kFacF32 ? 4 : 2);
                    if constexpr (MODE == kFacF32) u.fv[t * FI + i] = *(const u32x4_a4*)(base + fo[t * FI + i]);
                    else u.fv[t * FI + i] = *(const u32x4_a2*)(base + fo[t * FI + i]);
                }
            } else {
#pragma unroll
                for (int h = 0; h < 2; ++h) u.fd[t][h].load(fp[t], g.r, g.Kc, min(j0[t] + l16, r1), k + h * 32 + lg * 8);
            }
        }
    };
    auto multiply = [&](const Unit& u) {
        // (LDS operations of one wave execute in order: the previous unit's fragment reads are ahead of these writes)
#pragma unroll
        for (int i = 0; i < 2 * RT; ++i) *(u32x4*)(xs + (i * 8 + (lane >> 3)) * LR_P + (lane & 7) * 8) = u.x[i];
        if constexpr (L::STAGE_F) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int i = 0; i < FI; ++i) {
                    const int jr = i * (16 / FI) + (MODE == kFacF32 ? lane >> 4 : lane >> 3);
                    const uint32_t keep = in_job[t] && j0[t] + jr < g.r ? 0xffffffffu : 0u;      // ranks beyond r are zero
                    const u32x4 v = u.fv[t * FI + i];
                    bf16_t* d = fs + (t * 16 + jr) * LR_P;
                    if constexpr (MODE == kFacF32)
                        *(u32x2*)(d + (lane & 15) * 4) = u32x2{pack_bf16x2(__uint_as_float(v[0]), __uint_as_float(v[1])) & keep,
                                                               pack_bf16x2(__uint_as_float(v[2]), __uint_as_float(v[3])) & keep};
                    else
                        *(u32x4*)(d + (lane & 7) * 8) = u32x4{v[0] & keep, v[1] & keep, v[2] & keep, v[3] & keep};
                }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            bf16x8 x[RT];
#pragma unroll
            for (int i = 0; i < RT; ++i) x[i] = *(const bf16x8*)(xs + (i * 16 + l16) * LR_P + h * 32 + lg * 8);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                bf16x8 w;
                if constexpr (L::STAGE_F) {
                    w = *(const bf16x8*)(fs + (t * 16 + l16) * LR_P + h * 32 + lg * 8);
                } else {
                    const uint32_t keep = in_job[t] && j0[t] + l16 < g.r ? 0xffffffffu : 0u;
                    const u32x4 v = u.fd[t][h].get();
                    w = __builtin_bit_cast(bf16x8, u32x4{v[0] & keep, v[1] & keep, v[2] & keep, v[3] & keep});
                }
#pragma unroll
                for (int i = 0; i < RT; ++i) acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x[i], acc[i][t], 0, 0, 0);
            }
        }
    };
    const int all = (int)(g.Kc >> 6), per = b.splits > 1 ? (all + b.splits - 1) / b.splits : all;
    const int first = (int)blockIdx.y * per + wave, units = min(all, (int)blockIdx.y * per + per), last = units - 1;
    if (first < units) {
        Unit a, c;
        load(a, first);
#pragma unroll 1
        for (int u = first;;) {
            int nx = u + NW;
            load(c, nx < last ? nx : last);            // (past the end: fetched again, never used)
            multiply(a);
            if (nx >= units) break;
            u = nx;
            nx = u + NW;
            load(a, nx < last ? nx : last);
            multiply(c);
            if (nx >= units) break;
            u = nx;
        }
    }
    f32x4* red = (f32x4*)lr_lds;                        // [NW][RT * NT][64], over the (now dead) tiles
    __syncthreads();
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) red[(wave * (RT * NT) + i * NT + t) * 64 + lane] = acc[i][t];
    __syncthreads();
    for (int idx = tid; idx < RT * NT * 64; idx += 64 * NW) {
        f32x4 v = red[idx];
#pragma unroll
        for (int w = 1; w < NW; ++w) v += red[w * (RT * NT * 64) + idx];
        const int l = idx & 63, t = (idx >> 6) % NT, i = (idx >> 6) / NT;
        const int64_t m = row0 + i * 16 + (l & 15);
        if (t * 16 >= cols || m >= b.n_rows) continue;
        if (b.splits > 1) {
            *(f32x4*)(b.partial + ((int64_t)blockIdx.y * b.n_rows + m) * cols + t * 16 + 4 * (l >> 4)) = v;
            continue;
        }
        const int f = t * 16 >= rp ? 1 : 0;
        *(u32x2*)(g.T + f * g.t_step + m * g.ld_t + t * 16 - f * rp + 4 * (l >> 4)) =
            u32x2{pack_bf16x2(v[0] * g.scale, v[1] * g.scale), pack_bf16x2(v[2] * g.scale, v[3] * g.scale)};
    }
}

template <int MODE, int NT, int RT, int NW>
static int launch_lowrank_one(const LowRankBatch& b, unsigned blocks, hipStream_t stream) {
    constexpr size_t lds = LowRankLds<MODE, NT, RT, NW>::bytes;
    static std::atomic<bool> attr_set{false};   // the attribute call is idempotent: a race only repeats it
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute((const void*)lowrank_kernel<MODE, NT, RT, NW>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) {
            xq_set_error("lowrank: cannot raise the dynamic LDS limit: %s", hipGetErrorString(e));
            return XQ_ERR_LAUNCH;
        }
        attr_set = true;
    }
    lowrank_kernel<MODE, NT, RT, NW><<<dim3(blocks, (unsigned)b.splits), 64 * NW, lds, stream>>>(b);
    return XQ_OK;
}
template <int MODE, int RT, int NW>
static int launch_lowrank_nt(const LowRankBatch& b, int nt, unsigned blocks, hipStream_t stream) {
    switch (nt) {
        case 1: return launch_lowrank_one<MODE, 1, RT, NW>(b, blocks, stream);
        case 2: return launch_lowrank_one<MODE, 2, RT, NW>(b, blocks, stream);
        case 3: return launch_lowrank_one<MODE, 3, RT, 8>(b, blocks, stream);      // (two units of three factor tiles take more than 128 registers)
        default: return launch_lowrank_one<MODE, 4, RT, 8>(b, blocks, stream);
    }
}

// 16 rows and sixteen waves to a block until every compute unit has one, then 32 rows and eight waves
static bool lowrank_tall(int n, int64_t n_rows) { return n_rows * n > 16ll * num_cus(); }

int64_t lowrank_panel_bytes(int n, int64_t n_rows, int cols, int64_t Kc) {
    return lowrank_tall(n, n_rows) ? (((int64_t)cols * Kc * 2 + 255) & ~(int64_t)255) * n : 0;
}

// T[m][j] = bf16(scale * (partial[0][m][j] + partial[1][m][j] + ...)), the splits in index order; columns from rp on are the
// second product's
__global__ void __launch_bounds__(256) lowrank_reduce_kernel(const float* partial, int splits, int64_t n_rows, int rp, int nprod, float scale,
                                                             bf16_t* T, bf16_t* T2, int64_t ld_t) {
    const int cols = nprod * rp;
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x, total = n_rows * cols;
    if (t >= total) return;
    float v = partial[t];
    for (int s = 1; s < splits; ++s) v += partial[(int64_t)s * total + t];
    const int64_t m = t / cols;
    const int j = (int)(t - m * cols);
    (j < rp ? T : T2)[m * ld_t + (j < rp ? j : j - rp)] = to_bf16(v * scale);
}

// Splits of the contraction of one product where its blocks leave compute units idle.  A block pulls its rows and the whole factor
// through one compute unit, about 0.1 MB a microsecond; the launch that adds the splits' sums costs three.  us before and with splits: MLP
// 4096/12288 forward of 120 rows r 16 114 / 104, r 64 147 / 121, nvfp4 of 700 rows r 32 354 / 332; one projection [4096, 12288] forward and
// backward of 300 rows r 64 212 / 180, [12288, 4096] r 16 166 / 159; below the line (512 rows, K 4096, r 16) one launch is level or ahead.
static int lowrank_splits(const LowRankJob& j, int64_t blocks, FactorMode mode, const float* scratch, int64_t scratch_bytes, int64_t n_rows) {
    const int64_t bytes = j.Kc * (32 + (mode == kFacF32 || mode == kFacF32T ? 4 : 2) * (int64_t)j.nf * j.rp);
    int64_t s = std::min(num_cus() / blocks, j.Kc / 1024);      // (a unit of 64 for each of sixteen waves)
    if (s > 8) s = 8;
    if (s < 2 || bytes - bytes / s < 400000 || !xq_aligned(scratch, 16) || !scratch || scratch_bytes < s * n_rows * j.nf * j.rp * 4) return 1;
    return (int)s;
}

int launch_lowrank(const LowRankJob* jobs, int n, int64_t n_rows, FactorMode mode, bf16_t* panels, hipStream_t stream, float* scratch,
                   int64_t scratch_bytes) {
    XQ_REQUIRE(n >= 1 && n <= kLowRankJobs, "lowrank: %d products", n);
    if (n_rows == 0) return XQ_OK;
    LowRankBatch b{};
    const bool tall = lowrank_tall(n, n_rows);
    // every block reads the whole factor: where there are many, fp32 [r, K] factors are laid out as bf16 panels first (8192 rows,
    // K 4096, two factors of rank 32: 70 us against 40 and 6)
    LowRankJob own[kLowRankJobs];
    if (tall && mode == kFacF32 && panels) {
        PanelJobs pj{};
        pj.in_f32 = 1;
        for (int i = 0; i < n; ++i) {
            own[i] = jobs[i];
            for (int f = 0; f < jobs[i].nf; ++f)
                own[i].F[f] = pj.add(jobs[i].F[f], 1, jobs[i].r, jobs[i].Kc, false, panels + (int64_t)f * jobs[i].rp * jobs[i].Kc, 1, jobs[i].rp, jobs[i].Kc);
            own[i].r = jobs[i].rp;
            panels += (((int64_t)jobs[i].nf * jobs[i].rp * jobs[i].Kc * 2 + 255) & ~(int64_t)255) / 2;
        }
        const int rc = launch_panel_prep(pj, stream);
        if (rc) return rc;
        jobs = own;
        mode = kFacBf16;
    }
    const int64_t per = tall ? 32 : 16, blocks = xq_cdiv(n_rows, per);
    int nt = 1;
    for (int i = 0; i < n; ++i) {
        const LowRankJob& j = jobs[i];
        XQ_REQUIRE(j.rp > 0 && j.rp % 16 == 0 && j.r >= 1 && j.r <= j.rp && j.nf >= 1 && j.nf <= 2 && j.nf * j.rp <= 64, "lowrank: bad rank (r %d, r_pad %d)", j.r, j.rp);
        XQ_REQUIRE(j.Kc < (1ll << 24), "lowrank: contraction length %lld", (long long)j.Kc);
        XQ_REQUIRE(j.Kc % 64 == 0, "lowrank: contraction length %lld must be a multiple of 64", (long long)j.Kc);
        XQ_REQUIRE(j.ld_in % 8 == 0 && xq_aligned(j.In, 16), "lowrank: activation rows must be 16-byte aligned");
        XQ_REQUIRE(j.ld_t % 4 == 0 && j.t_step % 4 == 0 && xq_aligned(j.T, 8), "lowrank: result rows must be 8-byte aligned");
        b.job[i] = j;
        b.first[i] = (int32_t)(blocks * i);
        nt = j.nf * j.rp / 16 > nt ? j.nf * j.rp / 16 : nt;
    }
    b.n = n; b.n_rows = n_rows;
    b.splits = n == 1 && !tall ? lowrank_splits(jobs[0], blocks, mode, scratch, scratch_bytes, n_rows) : 1;
    b.partial = scratch;
    const unsigned grid = (unsigned)(blocks * n);
    int rc;
#define XQ_LR(MODE) rc = tall ? launch_lowrank_nt<MODE, 2, 8>(b, nt, grid, stream) : launch_lowrank_nt<MODE, 1, 16>(b, nt, grid, stream)
    switch (mode) {
        case kFacBf16: XQ_LR(kFacBf16); break;
        case kFacF32: XQ_LR(kFacF32); break;
        case kFacF32T: XQ_LR(kFacF32T); break;
        default: XQ_LR(kFacBf16T); break;
    }
#undef XQ_LR
    if (rc) return rc;
    XQ_CHECK_LAUNCH("lowrank");
    if (b.splits > 1) {
        const LowRankJob& j = jobs[0];
        lowrank_reduce_kernel<<<(unsigned)xq_cdiv(n_rows * j.nf * j.rp, 256), 256, 0, stream>>>(scratch, b.splits, n_rows, j.rp, j.nf, j.scale, j.T,
                                                                                                 j.T + j.t_step, j.ld_t);
        XQ_CHECK_LAUNCH("lowrank_reduce");
    }
    return XQ_OK;
}

// ------------------------------------------------------------------ SwiGLU backward + its two low-rank products
// One pass over (gate, up, dh): writes dgate | dup (the elementwise kernel's arithmetic, ops/moe/lora.py:855-917 with no
// routing weight) and forms Tg = s * dgate . Fg^T and Tu = s * dup . Fu^T from the values on their way out -- the two
// products do not read dgate | dup back.  Dense rows: 32 per block, the four waves (and blockIdx.y) split the columns, 64 at a
// time through wave-private LDS tiles.  A block of 32 rows runs ~140 us at 12288 columns however many there are, so a launch
// of fewer than a block per compute unit deals the columns over blockIdx.y too and leaves fp32 sums to
// lowrank_reduce_kernel (200 rows of 12288 columns: 141 us in 7 blocks, 18 us in 168 and the reduction).
struct SiluNtArgs {
    const bf16_t* gate;
    const bf16_t* up;
    int64_t ld_gu;
    const bf16_t* dh;
    int64_t ld_dh;
    bf16_t* dgate;
    bf16_t* dup;
    int64_t ld_out;
    int64_t n_rows, Kc;        // rows; columns of gate / up / dh (the contraction length of the two products)
    const void* Fg;            // factors in the kernel's MODE (routed rows: bf16 panels [r_pad][Kc] per expert)
    const void* Fu;
    int r, r_pad;
    float scale;
    bf16_t* Tg;                // [n_rows][ld_t]
    bf16_t* Tu;
    int64_t ld_t;
    // routed rows (GROUPED): rows in expert order, a factor pair per expert (stride 0: shared), the routing weight of a row
    // applied as the elementwise kernel applies it, and its gradient
    const int32_t* offsets;
    const int32_t* tile_offsets;
    int32_t num_experts;
    int64_t fg_stride, fu_stride;
    const float* row_w;
    float* d_row_w;
    float limit;               // SwiGLU limit on the gate pre-activation (<= 0: none)
    float* partial;            // dense with gridDim.y > 1: fp32 sums [gridDim.y][n_rows][products * r_pad]
};

// GROUPED: routed rows in expert order, organisation of small_nt_kernel<FJ> (a block = a 128-row tile of one expert, a
// wave = 32 rows over all columns, the expert's own factor pair), the routing weight applied and its gradient formed as
// the elementwise kernel does (the sum over a row runs in another order here: 16 lanes' partial sums, then a butterfly).
// FWD: the forward pass in the same organisation -- h = bf16(bf16(silu(gate)) * up) (routed: then rounded and times the row's
// weight), the elementwise forward kernel's arithmetic, written through `dgate`, and Tg = scale * h . Fg^T from the values
// on their way out (dh, dup, Fu, Tu, d_row_w unused).
// NARROW (GROUPED): 32 rows per block and the columns split over its eight waves, whose sums meet in LDS.  A wave's chunk is some 3 us of
// vector work beside its trip to memory, and in the wide form a wave walks all the columns: 64 us however few the rows (the launchers
// have both forms' times).
template <int FJ, bool GROUPED, bool FWD, int MODE, bool NARROW = false>
__global__ void __launch_bounds__(NARROW ? 512 : 256, NARROW ? 1 : 2) silu_bwd_nt_kernel(SiluNtArgs g) {
    static_assert(FJ <= 8, "one MFMA column tile per product");
    static_assert(GROUPED || !NARROW, "the narrow form is one of routed rows");
    constexpr int NW = NARROW ? 8 : 4;
    // 64 columns at a time (where small_nt_kernel takes 128: the same MFMA steps in the same order): three operands' pieces
    // are 12 KB per wave in flight, and two blocks share a compute unit
    constexpr int CW = 64, P = CW + 8;           // columns of a chunk; LDS row pitch (144 B: the 16 lanes of a read phase hit distinct banks)
    constexpr int NL = 32 * CW / 512;            // 16-byte loads per lane and operand chunk (a load instruction covers 512 / CW rows)
    constexpr int RPI = 512 / CW;                // rows per load instruction
    constexpr int FL = (FJ * 4 + RPI - 1) / RPI; // loads per lane of a factor chunk (FJ * 4 rows)
    constexpr int WTILE = (32 + 32) * P;         // bf16 elements per wave: value tile + factor tile
    extern __shared__ __attribute__((aligned(16))) bf16_t sn_lds[];
    __shared__ int sh_info[3];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int e = 0;
    int64_t row0, row_end;
    if constexpr (GROUPED) {
        // the expert whose tile range holds this block's tile: one look per thread, all loads in flight together
        if (tid == 0) sh_info[0] = -1;
        __syncthreads();
        const int t = NARROW ? blockIdx.x % (gridDim.x >> 2) : blockIdx.x;     // (a tile's four parts a stretch apart: experts of few rows fill only the first)
        for (int x = tid; x < g.num_experts; x += 64 * NW) {
            const int lo = g.tile_offsets[x], hi = g.tile_offsets[x + 1];
            const int o0 = g.offsets[x], o1 = g.offsets[x + 1];
            if (lo <= t && t < hi) {
                sh_info[0] = x;
                sh_info[1] = o0 + (t - lo) * 128;
                sh_info[2] = o1;
            }
        }
        __syncthreads();
        e = sh_info[0];
        if (e < 0) return;
        row0 = sh_info[1] + (NARROW ? (int)(blockIdx.x / (gridDim.x >> 2)) : wave) * 32;
        row_end = sh_info[2];
        if (row0 >= row_end) return;             // (a wave of the wide form: no block barrier from here on there)
    } else {
        row0 = (int64_t)blockIdx.x * 32;
        row_end = g.n_rows;
        if (row0 >= row_end) return;
    }
    const void* Fg = GROUPED ? (const void*)((const bf16_t*)g.Fg + (int64_t)e * g.fg_stride) : g.Fg;
    const void* Fu = GROUPED ? (const void*)((const bf16_t*)g.Fu + (int64_t)e * g.fu_stride) : g.Fu;
    bf16_t* xs = sn_lds + wave * WTILE;          // [32][P]
    bf16_t* fs = xs + 32 * P;                    // [32][P]
    const int fr = lane & 31, fk = (lane >> 5) * 8;
    const int crow = lane / (CW / 8), cpiece = (lane % (CW / 8)) * 8;
    const int frows = g.r_pad;
    // (dense: the 64-column units dealt evenly over the waves of the block column)
    const int64_t units = g.Kc / CW, parts = NW * gridDim.y, part = NW * blockIdx.y + wave;
    constexpr bool WHOLE = GROUPED && !NARROW;   // a wave takes all columns
    const int64_t kbeg = WHOLE ? 0 : units * part / parts * CW, kend = WHOLE ? g.Kc : units * (part + 1) / parts * CW;
    const int64_t rbase = row0 + crow;           // this lane's rows: rbase + RPI j, clamped onto the last row
    auto row_of = [&](int j) { const int64_t r = rbase + j * RPI; return r < row_end ? r : row_end - 1; };
    float rw[GROUPED ? NL : 1], wsum[GROUPED ? NL : 1];
    if constexpr (GROUPED) {
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            rw[j] = g.row_w[row_of(j)];
            wsum[j] = 0.0f;
        }
    }
    u32x4 gq[NL], uq[NL], dq[NL];
    FactorPiece<MODE> fq[FL];
    // every load is unconditional: rows past the end and pieces past the wave's columns are clamped onto valid ones
    auto fetch = [&](int64_t k) {
        int64_t kc = k + cpiece;
        kc = kc < kend ? kc : kend - 8;
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            const int64_t r = row_of(j);
            gq[j] = *(const u32x4*)(g.gate + r * g.ld_gu + kc);
            uq[j] = *(const u32x4*)(g.up + r * g.ld_gu + kc);
            if constexpr (!FWD) dq[j] = *(const u32x4*)(g.dh + r * g.ld_dh + kc);
        }
    };
    auto fetch_f = [&](const void* F, int64_t k) {
        int64_t kc = k + cpiece;
        kc = kc < kend ? kc : kend - 8;
#pragma unroll
        for (int j = 0; j < FL; ++j) fq[j].load(F, g.r, g.Kc, j * RPI + crow < g.r ? j * RPI + crow : g.r - 1, kc);
    };
    auto stage_f = [&]() {                       // ranks from r to the padded count are zero
        const u32x4 z = {0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < FL; ++j)
            if (j * RPI + crow < 32) *(u32x4*)(fs + (j * RPI + crow) * P + cpiece) = j * RPI + crow < g.r ? fq[j].get() : z;
    };
    f32x16 acc_g, acc_u;
#pragma unroll
    for (int q = 0; q < 16; ++q) acc_g[q] = acc_u[q] = 0.0f;
    auto multiply = [&](f32x16& acc, int nsteps) {
#pragma unroll
        for (int st = 0; st < CW / 16; ++st) {
            if (st < nsteps) {                   // uniform
                const bf16x8 a = *(const bf16x8*)(xs + fr * P + st * 16 + fk);
                const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
                const bf16x8 b = fr < frows ? *(const bf16x8*)(fs + fr * P + st * 16 + fk) : zero8;
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
            }
        }
    };
    // The factor chunks (from L2) are requested ahead of the value chunks and go to the LDS tile as soon as the MFMAs that
    // read its previous contents are issued (LDS operations of one wave execute in order), so their registers are free
    // while a chunk's values are worked out.
    if (kbeg < kend) {                           // (fewer units than waves: nothing to fetch)
        fetch_f(Fg, kbeg);
        fetch(kbeg);
        stage_f();
    }
    if constexpr (FWD) {
        for (int64_t k = kbeg; k < kend; k += CW) {
            const int64_t kc = k + cpiece;
            const bool mine = kc < kend;
#pragma unroll
            for (int j = 0; j < NL; ++j) {
                u32x4 oh;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float res[2];
#pragma unroll
                    for (int hlf = 0; hlf < 2; ++hlf) {
                        const float gv = swiglu_clamp(bf16_to_f32((bf16_t)(gq[j][i] >> (16 * hlf))), g.limit), uv = bf16_to_f32((bf16_t)(uq[j][i] >> (16 * hlf)));
                        const float a = round_bf16(gv * sigmoid_f32(gv));
                        float v = a * uv;
                        if constexpr (GROUPED) v = round_bf16(v) * rw[j];
                        res[hlf] = v;
                    }
                    oh[i] = pack_bf16x2(res[0], res[1]);
                }
                if (rbase + j * RPI < row_end && mine) *(u32x4*)(g.dgate + (rbase + j * RPI) * g.ld_out + kc) = oh;
                *(u32x4*)(xs + (j * RPI + crow) * P + cpiece) = oh;
            }
            fetch_f(Fg, k + CW);                // (past the last chunk: clamped, never used)
            fetch(k + CW);
            const int64_t left = kend - k;
            multiply(acc_g, (int)((left < CW ? left : CW) >> 4));
            stage_f();
        }
    } else
    for (int64_t k = kbeg; k < kend; k += CW) {
        const int64_t kc = k + cpiece;
        const bool mine = kc < kend;             // this lane's piece lies in the wave's columns
        fetch_f(Fu, k);
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            u32x4 og, ou;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float rg[2], ru[2];
#pragma unroll
                for (int hlf = 0; hlf < 2; ++hlf) {
                    const float g_raw = bf16_to_f32((bf16_t)(gq[j][i] >> (16 * hlf))), uv = bf16_to_f32((bf16_t)(uq[j][i] >> (16 * hlf)));
                    const float gv = swiglu_clamp(g_raw, g.limit), open = swiglu_mask(g_raw, g.limit);
                    const float d = bf16_to_f32((bf16_t)(dq[j][i] >> (16 * hlf)));
                    const float sg = sigmoid_f32(gv);
                    const float a = round_bf16(gv * sg);
                    float dp = d;
                    if constexpr (GROUPED) {
                        dp = round_bf16(d * rw[j]);
                        if (mine) wsum[j] += d * round_bf16(a * uv);
                    }
                    rg[hlf] = round_bf16(dp * uv) * (sg * (1.0f + gv * (1.0f - sg))) * open;
                    ru[hlf] = a * dp;
                }
                og[i] = pack_bf16x2(rg[0], rg[1]);
                ou[i] = pack_bf16x2(ru[0], ru[1]);
            }
            if (rbase + j * RPI < row_end && mine) {
                const int64_t r = rbase + j * RPI;
                *(u32x4*)(g.dgate + r * g.ld_out + kc) = og;
                *(u32x4*)(g.dup + r * g.ld_out + kc) = ou;
            }
            *(u32x4*)(xs + (j * RPI + crow) * P + cpiece) = og;
            uq[j] = ou;                          // waits in registers for its turn in the tile
        }
        const int64_t left = kend - k;
        const int nsteps = (int)((left < CW ? left : CW) >> 4);
        multiply(acc_g, nsteps);
#pragma unroll
        for (int j = 0; j < NL; ++j) *(u32x4*)(xs + (j * RPI + crow) * P + cpiece) = uq[j];
        stage_f();                               // the up factor's chunk
        fetch_f(Fg, k + CW);                    // (past the last chunk: clamped, never used)
        fetch(k + CW);
        multiply(acc_u, nsteps);
        stage_f();                               // the gate factor's next chunk
    }

    const int rgrp = (lane >> 5) * 4;
    if constexpr (GROUPED) {
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            float v = wsum[j];
#pragma unroll
            for (int o = 1; o < CW / 8; o <<= 1) v += __shfl_xor(v, o, 64);
            if (!NARROW && !FWD && g.d_row_w && lane % (CW / 8) == 0 && rbase + j * RPI < row_end) g.d_row_w[rbase + j * RPI] = v;
            wsum[j] = v;
        }
    }
    if constexpr (WHOLE) {
        if (fr < g.r_pad) {
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int64_t row = row0 + (q & 3) + rgrp + 8 * (q >> 2);
                if (row < row_end) {
                    g.Tg[row * g.ld_t + fr] = to_bf16(acc_g[q] * g.scale);
                    if constexpr (!FWD) g.Tu[row * g.ld_t + fr] = to_bf16(acc_u[q] * g.scale);
                }
            }
        }
        return;
    }
    // the waves' sums meet in LDS, in wave order
    constexpr int PR = FWD && NARROW ? 1 : 2;
    float* red = (float*)sn_lds;                 // [NW - 1 waves][PR products][16][64] floats, over the (now dead) tiles
    float* red_w = red + (NW - 1) * PR * 1024;   // NARROW: [NW][32] sums of the routing weights' gradients
    __syncthreads();
    if (wave > 0) {
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            red[(((wave - 1) * PR + 0) * 16 + q) * 64 + lane] = acc_g[q];
            if constexpr (PR > 1) red[(((wave - 1) * PR + 1) * 16 + q) * 64 + lane] = acc_u[q];
        }
    }
    if constexpr (NARROW && !FWD) {
        if (lane % (CW / 8) == 0) {
#pragma unroll
            for (int j = 0; j < NL; ++j) red_w[wave * 32 + j * RPI + crow] = wsum[j];
        }
    }
    __syncthreads();
    if constexpr (NARROW && !FWD) {
        if (wave == 1 && lane < 32 && g.d_row_w && row0 + lane < row_end) {
            float v = red_w[lane];
            for (int w = 1; w < NW; ++w) v += red_w[w * 32 + lane];
            g.d_row_w[row0 + lane] = v;
        }
    }
    if (wave > 0) return;
#pragma unroll
    for (int s = 1; s < NW; ++s)
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            acc_g[q] += red[(((s - 1) * PR + 0) * 16 + q) * 64 + lane];
            if constexpr (PR > 1) acc_u[q] += red[(((s - 1) * PR + 1) * 16 + q) * 64 + lane];
        }
    if (gridDim.y > 1) {
        constexpr int NP = 2;
        float* part_out = g.partial + (int64_t)blockIdx.y * g.n_rows * (NP * g.r_pad);
        if (fr < g.r_pad) {
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int64_t row = row0 + (q & 3) + rgrp + 8 * (q >> 2);
                if (row < row_end) {
                    part_out[row * (NP * g.r_pad) + fr] = acc_g[q];
                    part_out[row * (NP * g.r_pad) + g.r_pad + fr] = acc_u[q];
                }
            }
        }
        return;
    }
    if (fr < g.r_pad) {
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int64_t row = row0 + (q & 3) + rgrp + 8 * (q >> 2);
            if (row < row_end) {
                g.Tg[row * g.ld_t + fr] = to_bf16(acc_g[q] * g.scale);
                if constexpr (!FWD) g.Tu[row * g.ld_t + fr] = to_bf16(acc_u[q] * g.scale);
            }
        }
    }
}

template <int FJ, bool GROUPED, bool FWD, int MODE, bool NARROW = false>
static int launch_silu_nt_one(const SiluNtArgs& g, dim3 blocks, hipStream_t stream) {
    constexpr int NW = NARROW ? 8 : 4;
    constexpr size_t lds = (size_t)NW * (32 + 32) * (64 + 8) * 2;
    static std::atomic<bool> attr_set{false};   // the attribute call is idempotent: a race only repeats it
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute((const void*)silu_bwd_nt_kernel<FJ, GROUPED, FWD, MODE, NARROW>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) {
            xq_set_error("silu_bwd_nt: cannot raise the dynamic LDS limit: %s", hipGetErrorString(e));
            return XQ_ERR_LAUNCH;
        }
        attr_set = true;
    }
    silu_bwd_nt_kernel<FJ, GROUPED, FWD, MODE, NARROW><<<blocks, 64 * NW, lds, stream>>>(g);
    XQ_CHECK_LAUNCH("silu_bwd_nt");
    return XQ_OK;
}

bool silu_bwd_nt_supported(int64_t cols, int r_pad) { return (r_pad == 16 || r_pad == 32) && cols % 64 == 0 && cols >= 512; }

// column splits of the dense form: none from a block per compute unit on, else about three blocks per unit, 512 columns at least
static int silu_nt_splits(int64_t n_rows, int64_t cols) {
    const int64_t blocks = xq_cdiv(n_rows, 32);
    if (blocks >= num_cus()) return 1;
    int64_t s = xq_cdiv(3ll * num_cus(), blocks);
    if (s > cols / 512) s = cols / 512;
    return s < 2 ? 1 : (int)s;
}

int64_t silu_nt_partial_bytes(int64_t n_rows, int64_t cols, int r_pad) {
    const int s = n_rows > 0 ? silu_nt_splits(n_rows, cols) : 1;
    return s > 1 ? (int64_t)s * n_rows * 2 * r_pad * 4 : 0;
}

int launch_silu_bwd_nt(const bf16_t* gate, const bf16_t* up, int64_t ld_gu, const bf16_t* dh, int64_t ld_dh, bf16_t* dgate,
                       bf16_t* dup, int64_t ld_out, int64_t n_rows, int64_t cols, const void* Fg, const void* Fu, FactorMode mode, int r, int r_pad,
                       float scale, bf16_t* Tg, bf16_t* Tu, int64_t ld_t, float* partial, hipStream_t stream, const int32_t* offsets,
                       const int32_t* tile_offsets, int32_t num_experts, bool shared_fg, bool shared_fu, const float* row_w,
                       float* d_row_w, float swiglu_limit) {
    XQ_REQUIRE(silu_bwd_nt_supported(cols, r_pad), "silu_bwd_nt: %lld columns with r_pad %d are not handled here", (long long)cols, r_pad);
    XQ_REQUIRE(ld_gu % 8 == 0 && ld_dh % 8 == 0 && ld_out % 8 == 0 && ld_t >= r_pad, "silu_bwd_nt: row pitches must be multiples of 8");
    XQ_REQUIRE(xq_aligned(gate, 16) && xq_aligned(up, 16) && xq_aligned(dh, 16) && xq_aligned(dgate, 16) && xq_aligned(dup, 16),
               "silu_bwd_nt: operands must be 16-byte aligned");
    XQ_REQUIRE(!offsets || (tile_offsets && row_w && num_experts >= 1), "silu_bwd_nt: the routed form needs tile offsets and row weights");
    if (n_rows == 0) return XQ_OK;
    SiluNtArgs g{gate, up, ld_gu, dh, ld_dh, dgate, dup, ld_out, n_rows, cols, Fg, Fu, r, r_pad, scale, Tg, Tu, ld_t,
                 offsets, tile_offsets, num_experts, offsets && !shared_fg ? (int64_t)r_pad * cols : 0,
                 offsets && !shared_fu ? (int64_t)r_pad * cols : 0, row_w, d_row_w, swiglu_limit, nullptr};
    if (offsets) {
        XQ_REQUIRE(mode == kFacBf16, "silu_bwd_nt: the routed form takes bf16 panels");
        const dim3 blocks((unsigned)(xq_cdiv(n_rows, 128) + num_experts));
        if (n_rows <= 64ll * num_cus()) {        // (us, wide -> narrow, 64 experts of 1024 columns, r 16: 1800 rows 64 -> 19, 12000 70 -> 43, 24000 78 -> 79)
            const dim3 four(4 * blocks.x);
            return r_pad == 16 ? launch_silu_nt_one<4, true, false, kFacBf16, true>(g, four, stream) : launch_silu_nt_one<8, true, false, kFacBf16, true>(g, four, stream);
        }
        return r_pad == 16 ? launch_silu_nt_one<4, true, false, kFacBf16>(g, blocks, stream) : launch_silu_nt_one<8, true, false, kFacBf16>(g, blocks, stream);
    }
    XQ_REQUIRE(mode != kFacF32, "silu_bwd_nt: factor form %d", (int)mode);
    const int splits = partial ? silu_nt_splits(n_rows, cols) : 1;
    g.partial = splits > 1 ? partial : nullptr;
    const dim3 blocks((unsigned)xq_cdiv(n_rows, 32), (unsigned)splits);
    int rc;
#define XQ_SILU(MODE) rc = r_pad == 16 ? launch_silu_nt_one<4, false, false, MODE>(g, blocks, stream) : launch_silu_nt_one<8, false, false, MODE>(g, blocks, stream)
    if (mode == kFacBf16) XQ_SILU(kFacBf16);
    else if (mode == kFacF32T) XQ_SILU(kFacF32T);
    else XQ_SILU(kFacBf16T);
#undef XQ_SILU
    if (rc || splits == 1) return rc;
    lowrank_reduce_kernel<<<(unsigned)xq_cdiv(n_rows * 2 * r_pad, 256), 256, 0, stream>>>(partial, splits, n_rows, r_pad, 2, scale, Tg, Tu, ld_t);
    XQ_CHECK_LAUNCH("silu_bwd_nt(reduce)");
    return XQ_OK;
}

int launch_silu_fwd_nt(const bf16_t* gate, const bf16_t* up, int64_t ld_gu, bf16_t* h, int64_t ld_h, int64_t n_rows, int64_t cols,
                       const bf16_t* F, int r_pad, float scale, bf16_t* T, int64_t ld_t, hipStream_t stream, const int32_t* offsets,
                       const int32_t* tile_offsets, int32_t num_experts, bool shared_f, const float* row_w, float swiglu_limit) {
    XQ_REQUIRE(silu_bwd_nt_supported(cols, r_pad), "silu_fwd_nt: %lld columns with r_pad %d are not handled here", (long long)cols, r_pad);
    XQ_REQUIRE(ld_gu % 8 == 0 && ld_h % 8 == 0 && ld_t >= r_pad, "silu_fwd_nt: row pitches must be multiples of 8");
    XQ_REQUIRE(xq_aligned(gate, 16) && xq_aligned(up, 16) && xq_aligned(h, 16) && xq_aligned(F, 16), "silu_fwd_nt: operands must be 16-byte aligned");
    XQ_REQUIRE(!offsets || (tile_offsets && row_w && num_experts >= 1), "silu_fwd_nt: the routed form needs tile offsets and row weights");
    if (n_rows == 0) return XQ_OK;
    SiluNtArgs g{gate, up, ld_gu, nullptr, 0, h, nullptr, ld_h, n_rows, cols, F, F, r_pad, r_pad, scale, T, nullptr, ld_t,
                 offsets, tile_offsets, num_experts, offsets && !shared_f ? (int64_t)r_pad * cols : 0, 0, row_w, nullptr, swiglu_limit, nullptr};
    if (!offsets) {
        const dim3 blocks((unsigned)xq_cdiv(n_rows, 32));
        return r_pad == 16 ? launch_silu_nt_one<4, false, true, kFacBf16>(g, blocks, stream) : launch_silu_nt_one<8, false, true, kFacBf16>(g, blocks, stream);
    }
    const dim3 blocks((unsigned)(xq_cdiv(n_rows, 128) + num_experts));
    if (n_rows <= (r_pad == 16 ? 160ll : 64ll) * num_cus()) {      // (the same: 1800 rows 32 -> 15, 12000 40 -> 22, 24000 46 -> 38, 48000 65 -> 66; r 32: 16000 57 -> 45, 24000 of 896 columns 3 us behind)
        const dim3 four(4 * blocks.x);
        return r_pad == 16 ? launch_silu_nt_one<4, true, true, kFacBf16, true>(g, four, stream) : launch_silu_nt_one<8, true, true, kFacBf16, true>(g, four, stream);
    }
    return r_pad == 16 ? launch_silu_nt_one<4, true, true, kFacBf16>(g, blocks, stream) : launch_silu_nt_one<8, true, true, kFacBf16>(g, blocks, stream);
}

// ------------------------------------------------------------------ tn (weight-gradient shape)
struct TnArgs {
    const bf16_t* P;
    int64_t ldp;
    int64_t width;
    const bf16_t* Q;
    int r_pad, r_out;
    int64_t n_rows;
    int64_t rows_per_split;
    int transpose_out;
    float* out;              // dense: partial [S][width][r_pad]; grouped: out [E][...]
    const int32_t* offsets;  // grouped
    const int32_t* row_limit;  // dense, optional (device): only rows below *row_limit are contracted
    int64_t ldq;               // row pitch of Q in elements
    const int32_t* p_rows;     // optional: row m of the contraction is row p_rows[m] of P
    float* out2;               // optional: columns of Q from split_j on belong to a second result, columns split_j .. + r_out
    int32_t split_j;
};

constexpr int TN_PP = 128 + 16;  // Ps pitch (bf16 elements): 288 B rows
constexpr int TN_QP = 80;        // Qs pitch: 160 B rows

constexpr int TN_CHUNK = 1024;   // grouped: rows per block (global row chunks, cut at expert boundaries)

// acc += P[m_begin:m_end, c0 + wave*32 .. +32]^T . Q[m_begin:m_end, :]  (m_begin < m_end).  Rows go through LDS 32 at
// a time, in two alternating buffers (Ps, Qs hold both), so one block barrier per tile is enough; the tiles m + 64
// and m + 96 are in flight in registers while tiles m and m + 32 are multiplied.  Every load is unconditional:
// rows past m_end are clamped onto the last row and their Q values replaced by zero, columns past the width are
// clamped onto column 0 and never written.
template <int NT>
__device__ __forceinline__ void tn_accumulate(const TnArgs& g, int64_t c0, int64_t m_begin, int64_t m_end, bf16_t* Ps,
                                              bf16_t* Qs, f32x16* acc) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int pr = tid >> 4, pc = (tid & 15) * 8;  // P tile: rows pr, pr+16; 8 cols at pc
    const int64_t pcol = c0 + pc < g.width ? c0 + pc : 0;   // width % 8 == 0
    const int qchunks = g.r_pad / 8;
    const bool q_thread = tid < 32 * qchunks;
    const int qr = q_thread ? tid / qchunks : 0, qc = q_thread ? (tid % qchunks) * 8 : 0;
    const u32x4 z = {0, 0, 0, 0};
    const int64_t last = m_end - 1;
    struct Tile { u32x4 p0, p1, q; int32_t i0, i1; };
    // with a row map, the P rows of tile m are named by entries fetched one stage earlier (with the data of tile m - 64):
    // the data loads then follow their indices without a round trip of their own in the steady state
    auto fetch_rows = [&](Tile& t, int64_t m) {
        if (g.p_rows) {
            const int64_t r0 = m + pr < m_end ? m + pr : last, r1 = m + pr + 16 < m_end ? m + pr + 16 : last;
            t.i0 = g.p_rows[r0];
            t.i1 = g.p_rows[r1];
        }
    };
    auto fetch = [&](Tile& t, int64_t m) {
        int64_t r0 = m + pr < m_end ? m + pr : last, r1 = m + pr + 16 < m_end ? m + pr + 16 : last;
        const int64_t rq = m + qr < m_end ? m + qr : last;
        if (g.p_rows) { r0 = t.i0; r1 = t.i1; }
        t.p0 = *(const u32x4*)(g.P + r0 * g.ldp + pcol);
        t.p1 = *(const u32x4*)(g.P + r1 * g.ldp + pcol);
        t.q = *(const u32x4*)(g.Q + rq * g.ldq + qc);
        fetch_rows(t, m + 64);
    };
    auto tile = [&](Tile& t, int64_t m, int buf) {     // multiply tile m out of LDS buffer `buf`, refill t with tile m + 64
        bf16_t* ps = Ps + buf * (32 * TN_PP);
        bf16_t* qs = Qs + buf * (32 * TN_QP);
        *(u32x4*)(ps + pr * TN_PP + pc) = t.p0;
        *(u32x4*)(ps + (pr + 16) * TN_PP + pc) = t.p1;
        if (q_thread) *(u32x4*)(qs + qr * TN_QP + qc) = m + qr < m_end ? t.q : z;
        fetch(t, m + 64);
        // the other buffer's fragment reads lie before this barrier in every wave, its next stores after the next one
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            bf16x8 a = lds_tr_frag(ps, TN_PP, ks * 16, wave * 32, lane);
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                bf16x8 b = lds_tr_frag(qs, TN_QP, ks * 16, n * 32, lane);
                acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[n], 0, 0, 0);
            }
        }
    };
    Tile ta, tb;
    fetch_rows(ta, m_begin);
    fetch_rows(tb, m_begin + 32);
    fetch(ta, m_begin);
    fetch(tb, m_begin + 32);
    for (int64_t m = m_begin; m < m_end; m += 64) {
        tile(ta, m, 0);
        tile(tb, m + 32, 1);        // past m_end: all-zero Q rows, no contribution
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // the buffers are free again when this returns
}

// out[c][j] (pitch = row length of the destination) or, transposed, out[j][c]; j < r_lim.  out2 (may be NULL): the columns from
// split_j on are that matrix's columns 0 ..
template <int NT>
__device__ __forceinline__ void tn_write(const f32x16* acc, float* out, int64_t c0, int64_t width, int r_lim, int pitch,
                                         bool transposed, float* out2 = nullptr, int split_j = 0) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int rgrp = (lane >> 5) * 4;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        int j = n * 32 + (lane & 31);
        if (out2 != nullptr && j >= split_j) { out = out2; j -= split_j; }
        if (j >= r_lim) continue;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int64_t c = c0 + wave * 32 + (q & 3) + rgrp + 8 * (q >> 2);
            if (c >= width) continue;
            if (transposed) out[(int64_t)j * width + c] = acc[n][q];
            else out[c * pitch + j] = acc[n][q];
        }
    }
}

// dense, up to kTnJobs products in one launch: block (job, col tile, row split) -> partial[split][width][r_pad], or the result
// itself where a job's rows are not split
struct TnBatch {
    TnArgs job[kTnJobs];
    float* partial[kTnJobs];
    int32_t first[kTnJobs + 1];       // first block of a job
    int32_t splits[kTnJobs];
    int32_t n;
};
template <int NT>
__global__ void __launch_bounds__(256) tn_kernel(TnBatch b) {
    __shared__ __attribute__((aligned(16))) bf16_t Ps[2 * 32 * TN_PP];
    __shared__ __attribute__((aligned(16))) bf16_t Qs[2 * 32 * TN_QP];
    int ji = 0;
#pragma unroll
    for (int i = 1; i < kTnJobs; ++i)
        if (i < b.n && (int)blockIdx.x >= b.first[i]) ji = i;
    const TnArgs& g = b.job[ji];
    const int splits = b.splits[ji], at = (int)blockIdx.x - b.first[ji], ct = at / splits, split = at - ct * splits;
    const int64_t c0 = (int64_t)ct * 128;
    const int64_t m_begin = (int64_t)split * g.rows_per_split;
    int64_t m_end = m_begin + g.rows_per_split;
    m_end = m_end < g.n_rows ? m_end : g.n_rows;
    if (g.row_limit) {
        const int64_t lim = *g.row_limit;
        m_end = m_end < lim ? m_end : lim;
    }
    f32x16 acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[n][q] = 0.0f;
    if (m_begin < m_end) tn_accumulate<NT>(g, c0, m_begin, m_end, Ps, Qs, acc);     // uniform over the block
    if (splits == 1) tn_write<NT>(acc, g.out, c0, g.width, g.r_out, g.r_out, g.transpose_out != 0, g.out2, g.split_j);
    else tn_write<NT>(acc, b.partial[ji] + (int64_t)split * g.width * g.r_pad, c0, g.width, g.r_pad, g.r_pad, false);
}

// grouped, up to kTnJobs products of the same rows in one launch: block (job, row part, col tile)
struct TnGroupedBatch {
    TnArgs job[kTnJobs];
    float* partial[kTnJobs];
    int32_t first[kTnJobs];           // first block of a job
    int32_t col_tiles[kTnJobs];
    int32_t n;
};
__device__ __forceinline__ int tn_grouped_job(const TnGroupedBatch& b, int* part, int64_t* c0) {
    int ji = 0;
#pragma unroll
    for (int i = 1; i < kTnJobs; ++i)
        if (i < b.n && (int)blockIdx.x >= b.first[i]) ji = i;
    const int at = (int)blockIdx.x - b.first[ji];
    *part = at / b.col_tiles[ji];
    *c0 = (int64_t)(at - *part * b.col_tiles[ji]) * 128;
    return ji;
}
template <int NT>
__device__ __forceinline__ void tn_write_expert(const TnArgs& g, const f32x16* acc, int64_t c0, int e) {
    const int64_t at = (int64_t)e * g.width * g.r_out;
    tn_write<NT>(acc, g.out + at, c0, g.width, g.r_out, g.r_out, g.transpose_out != 0, g.out2 ? g.out2 + at : nullptr, g.split_j);
}

// the expert that holds row `row` and the one before it (offsets[e] < row < offsets[e + 1]), -1 if a new expert, or none, starts
// there; one look per thread, the same answer in the whole block
__device__ __forceinline__ int tn_owner_across(const int32_t* offsets, int num_experts, int64_t row) {
    __shared__ int sh;
    if (threadIdx.x == 0) sh = -1;
    __syncthreads();
    for (int x = threadIdx.x; x < num_experts; x += 256)
        if (offsets[x] < row && row < offsets[x + 1]) sh = x;
    __syncthreads();
    return sh;
}

// experts of few rows on average: a block takes one expert's rows within one chunk of TN_CHUNK global rows.  Part e < E: expert
// e's first piece (written as the result where it is the only one, zero for an expert without rows); part E + c - 1: the piece
// with which the expert that crosses into chunk c goes on there.  Pieces, their places and the order of their sum are those of
// tn_grouped_kernel below: the same bits.
template <int NT>
__global__ void __launch_bounds__(256) tn_piece_kernel(TnGroupedBatch b, int32_t num_experts) {
    __shared__ __attribute__((aligned(16))) bf16_t Ps[2 * 32 * TN_PP];
    __shared__ __attribute__((aligned(16))) bf16_t Qs[2 * 32 * TN_QP];
    int part;
    int64_t c0;
    const int ji = tn_grouped_job(b, &part, &c0);
    const TnArgs& g = b.job[ji];
    const bool first = part < num_experts;
    const int e = first ? part : tn_owner_across(g.offsets, num_experts, (int64_t)(part - num_experts + 1) * TN_CHUNK);
    if (e < 0) return;
    const int64_t m_begin = first ? (int64_t)g.offsets[e] : (int64_t)(part - num_experts + 1) * TN_CHUNK;
    const int64_t ee = g.offsets[e + 1], chunk = m_begin / TN_CHUNK, chunk_end = (chunk + 1) * TN_CHUNK;
    const int64_t m_end = ee < chunk_end ? ee : chunk_end;
    f32x16 acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[n][q] = 0.0f;
    if (m_begin < m_end) tn_accumulate<NT>(g, c0, m_begin, m_end, Ps, Qs, acc);     // uniform over the block
    if (first && ee <= chunk_end) tn_write_expert<NT>(g, acc, c0, e);
    else tn_write<NT>(acc, b.partial[ji] + (chunk * 2 + (first ? 1 : 0)) * g.width * g.r_pad, c0, g.width, g.r_pad, g.r_pad, false);
}

// row part = chunk of TN_CHUNK global rows.  The chunk is walked expert by expert;
// an expert that lies wholly inside the chunk is written to out[e] directly, a piece of an expert
// that continues from the previous chunk goes to partial[chunk][0], one that continues into the
// next chunk to partial[chunk][1] (tn_grouped_reduce_kernel adds the pieces in chunk order).
// What bounds it: the rows in flight (two tiles of 32 a block).  A product of 131072 rows and 768 columns is 768 blocks, three a
// compute unit; the joint launch keeps the five that fit there to the end:
// the five products of 131072 rows (2048 and 768 columns, rank 16, gate and up side by side) 356 us one by one, 322 together.
template <int NT>
__global__ void __launch_bounds__(256) tn_grouped_kernel(TnGroupedBatch b, int32_t num_experts) {
    __shared__ __attribute__((aligned(16))) bf16_t Ps[2 * 32 * TN_PP];
    __shared__ __attribute__((aligned(16))) bf16_t Qs[2 * 32 * TN_QP];
    __shared__ int sh_e;
    int chunk;
    int64_t c0;
    const int ji = tn_grouped_job(b, &chunk, &c0);
    const TnArgs& g = b.job[ji];
    const int64_t r_begin = (int64_t)chunk * TN_CHUNK;
    int64_t r_end = r_begin + TN_CHUNK;
    r_end = r_end < g.n_rows ? r_end : g.n_rows;
    // the expert that owns row r_begin (offsets[e] <= r_begin < offsets[e + 1]; r_begin < n_rows = offsets[E], so
    // exactly one does): one look per thread instead of a chain of dependent loads
    if (threadIdx.x == 0) sh_e = num_experts;      // rows beyond the last expert's: nothing to do
    __syncthreads();
    for (int x = threadIdx.x; x < num_experts; x += 256) {
        const int64_t o0 = g.offsets[x], o1 = g.offsets[x + 1];
        if (o0 <= r_begin && r_begin < o1) sh_e = x;
    }
    __syncthreads();
    int e = sh_e;
    int64_t m = r_begin;
    while (m < r_end && e < num_experts) {
        const int64_t eb = g.offsets[e], ee = g.offsets[e + 1];
        const int64_t seg_end = ee < r_end ? ee : r_end;
        if (seg_end <= m) { ++e; continue; }   // expert without rows (or already passed)
        f32x16 acc[NT];
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[n][q] = 0.0f;
        tn_accumulate<NT>(g, c0, m, seg_end, Ps, Qs, acc);
        if (eb >= r_begin && ee <= r_end)
            tn_write_expert<NT>(g, acc, c0, e);
        else
            tn_write<NT>(acc, b.partial[ji] + ((int64_t)chunk * 2 + (eb < r_begin ? 0 : 1)) * g.width * g.r_pad, c0, g.width,
                         g.r_pad, g.r_pad, false);
        m = seg_end;
        ++e;
    }
}

// Four elements from t on of expert e's result: the sum of its pieces in chunk order, zero without rows
__device__ __forceinline__ void tn_reduce_expert(const TnArgs& g, const float* partial, int e, int64_t rb, int64_t en, int64_t t) {
    const int64_t c = t / g.r_pad;
    int j = (int)(t - c * g.r_pad);      // (r_pad and split_j are multiples of 16: the four lie in one row of one result)
    f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
    if (en > rb) {
        const int64_t ch0 = rb / TN_CHUNK, ch1 = (en - 1) / TN_CHUNK, per = g.width * g.r_pad;
        s = *(const f32x4*)(partial + (ch0 * 2 + 1) * per + t);
        for (int64_t ch = ch0 + 1; ch <= ch1; ++ch) s += *(const f32x4*)(partial + (ch * 2) * per + t);
    }
    float* o = g.out;
    if (g.out2 != nullptr && j >= g.split_j) { o = g.out2; j -= g.split_j; }
    o += (int64_t)e * g.width * g.r_out;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        if (j + u >= g.r_out) break;
        if (g.transpose_out) o[(int64_t)(j + u) * g.width + c] = s[u];
        else o[c * g.r_out + j + u] = s[u];
    }
}

// out[e] for the experts the chunk walk did not finish: zero for an expert without rows, the sum of
// its pieces in chunk order for one that spans several chunks.  Block x: 1024 elements of a job's [width, r_pad], y: expert
// (most blocks find their expert finished: four elements a thread keep their number down: 28 us for those five products,
// 55 with one element).  CROSS, behind tn_piece_kernel, which has finished every expert within one chunk and those without
// rows: y: the boundary before chunk y + 1, for the expert that crosses it as its first.
template <bool CROSS>
__global__ void __launch_bounds__(256) tn_grouped_reduce_kernel(TnGroupedBatch b, int32_t num_experts) {
    int ji = 0;
#pragma unroll
    for (int i = 1; i < kTnJobs; ++i)
        if (i < b.n && (int)blockIdx.x >= b.first[i]) ji = i;
    const TnArgs& g = b.job[ji];
    const int64_t boundary = (int64_t)(blockIdx.y + 1) * TN_CHUNK;
    const int e = CROSS ? tn_owner_across(g.offsets, num_experts, boundary) : (int)blockIdx.y;
    if (e < 0) return;
    const int64_t rb = g.offsets[e], en = g.offsets[e + 1];
    if constexpr (CROSS) {
        if (rb < boundary - TN_CHUNK) return;       // it has crossed one before
    } else {
        if (en > rb && rb / TN_CHUNK == (en - 1) / TN_CHUNK) return;   // written directly
    }
    const int64_t t = ((int64_t)((int)blockIdx.x - b.first[ji]) * 256 + threadIdx.x) * 4;
    if (t < g.width * g.r_pad) tn_reduce_expert(g, b.partial[ji], e, rb, en, t);
}

// sums the dense partials of up to kTnJobs products in split order: out[c][j] or out[j][c], j < r_out
struct TnReduceBatch {
    const float* partial[kTnJobs];
    float* out[kTnJobs];
    float* out2[kTnJobs];
    int64_t width[kTnJobs];
    int32_t splits[kTnJobs], r_pad[kTnJobs], r_out[kTnJobs], transpose_out[kTnJobs], split_j[kTnJobs];
    int32_t first[kTnJobs];
    int32_t n;
};
__global__ void __launch_bounds__(256) tn_reduce_kernel(TnReduceBatch b) {
    int ji = 0;
#pragma unroll
    for (int i = 1; i < kTnJobs; ++i)
        if (i < b.n && (int)blockIdx.x >= b.first[i]) ji = i;
    const int64_t t = (int64_t)((int)blockIdx.x - b.first[ji]) * 256 + threadIdx.x, width = b.width[ji];
    const int r_pad = b.r_pad[ji], r_out = b.r_out[ji];
    if (t >= width * r_pad) return;
    // (consecutive threads write along the destination's rows)
    int64_t c, j;
    if (b.transpose_out[ji]) { j = t / width; c = t - j * width; }
    else { c = t / r_pad; j = t - c * r_pad; }
    float s = 0.0f;
    const float* p = b.partial[ji] + c * r_pad + j;
    for (int i = 0; i < b.splits[ji]; ++i) s += p[(int64_t)i * width * r_pad];
    float* out = b.out[ji];
    if (b.out2[ji] != nullptr && j >= b.split_j[ji]) { out = b.out2[ji]; j -= b.split_j[ji]; }
    if (j >= r_out) return;
    if (b.transpose_out[ji]) out[j * width + c] = s;
    else out[c * r_out + j] = s;
}

// Row splits of `col_tiles` column tiles: about three blocks per compute unit, 512 rows each at least (below 1024 rows the
// second launch that sums the splits costs more than the split saves)
static int tn_splits(int64_t n_rows, int64_t col_tiles) {
    int64_t s = xq_cdiv(768, col_tiles);
    const int64_t max_s = n_rows / 512 > 0 ? n_rows / 512 : 1;
    if (s > max_s) s = max_s;
    if (s > 32) s = 32;
    return (int)(s < 1 ? 1 : s);
}

int64_t tn_partial_bytes(int64_t n_rows, int64_t width, int r_pad) {
    const int64_t dense = (int64_t)tn_splits(n_rows, xq_cdiv(width, 128)) * width * r_pad * 4;      // (a joint launch splits less)
    const int64_t grouped = xq_cdiv(n_rows > 0 ? n_rows : 1, TN_CHUNK) * 2 * width * r_pad * 4;
    const int64_t b = dense > grouped ? dense : grouped;
    return (b + 255) & ~(int64_t)255;
}

static int tn_check(const bf16_t* P, int64_t ldp, int64_t width, const bf16_t* Q, int64_t ldq, int r_pad, int r_out) {
    XQ_REQUIRE(ldq >= r_pad && ldq % 8 == 0, "tn: Q pitch %lld must be a multiple of 8 and at least r_pad", (long long)ldq);
    XQ_REQUIRE(r_pad > 0 && r_pad <= 64 && r_pad % 16 == 0 && r_out <= r_pad, "tn: bad rank (r_pad %d, r_out %d)", r_pad, r_out);
    XQ_REQUIRE(width % 8 == 0 && ldp % 8 == 0 && xq_aligned(P, 16) && xq_aligned(Q, 16), "tn: operands must be 16-byte aligned, width %% 8 == 0");
    return XQ_OK;
}

int launch_tn_multi(const TnJob* jobs, int n, int64_t n_rows, float* partial, hipStream_t stream, const int32_t* row_limit) {
    XQ_REQUIRE(n >= 0 && n <= kTnJobs, "tn: %d products", n);
    XQ_REQUIRE(partial != nullptr, "tn: partial workspace is NULL");
    TnBatch b{};
    TnReduceBatch rb{};
    int64_t col_tiles = 0;
    for (int i = 0; i < n; ++i) col_tiles += xq_cdiv(jobs[i].width, 128);
    const int S = col_tiles > 0 ? tn_splits(n_rows, col_tiles) : 1;
    const int64_t rps = xq_cdiv(xq_cdiv(n_rows, S), 32) * 32;
    int nt = 1;
    int64_t blocks = 0, rblocks = 0;
    for (int i = 0; i < n; ++i) {
        const TnJob& j = jobs[i];
        const int64_t ldq = j.ldq > 0 ? j.ldq : j.r_pad;
        const int rc = tn_check(j.P, j.ldp, j.width, j.Q, ldq, j.r_pad, j.r_out);
        if (rc) return rc;
        if (j.width == 0 || j.r_out == 0) continue;
        const int k = b.n++;
        b.job[k] = TnArgs{j.P, j.ldp, j.width, j.Q, j.r_pad, j.r_out, n_rows, rps, j.transpose_out ? 1 : 0, j.out, nullptr, row_limit, ldq, j.p_rows, j.out2, j.split_j};
        b.partial[k] = partial;
        b.splits[k] = S;
        b.first[k] = (int32_t)blocks;
        blocks += xq_cdiv(j.width, 128) * S;
        if (j.r_pad > 32) nt = 2;
        rb.partial[k] = partial; rb.out[k] = j.out; rb.out2[k] = j.out2; rb.width[k] = j.width; rb.splits[k] = S;
        rb.r_pad[k] = j.r_pad; rb.r_out[k] = j.r_out; rb.transpose_out[k] = j.transpose_out ? 1 : 0; rb.split_j[k] = j.split_j;
        rb.first[k] = (int32_t)rblocks;
        rblocks += xq_cdiv(j.width * j.r_pad, 256);
        partial += tn_partial_bytes(n_rows, j.width, j.r_pad) / 4;
    }
    if (b.n == 0) return XQ_OK;
    if (nt == 1) tn_kernel<1><<<(unsigned)blocks, 256, 0, stream>>>(b);
    else tn_kernel<2><<<(unsigned)blocks, 256, 0, stream>>>(b);
    XQ_CHECK_LAUNCH("tn");
    if (S > 1) {
        rb.n = b.n;
        tn_reduce_kernel<<<(unsigned)rblocks, 256, 0, stream>>>(rb);
        XQ_CHECK_LAUNCH("tn_reduce");
    }
    return XQ_OK;
}

int launch_tn_grouped_multi(const TnJob* jobs, int n, int64_t n_rows, float* partial, const int32_t* offsets, int32_t num_experts,
                            hipStream_t stream) {
    XQ_REQUIRE(n >= 0 && n <= kTnJobs, "tn: %d products", n);
    XQ_REQUIRE(partial != nullptr, "tn: partial workspace is NULL");
    // up to 256 rows an expert on average the experts of a column tile run side by side, a block for each (and for each further
    // chunk of one that spans several); beyond, a block walks a chunk of the row range expert by expert.
    // Backward of 128 block-fp8 experts [2048, 768], rank 16, us, walked chunks / blocks of an expert and chunk / one block an expert
    // whatever its rows: Zipf(1.1) loads of 4 rows an expert on average 603 / 345 / 345, of 64 505 / 455 / 448, of 256 (the largest
    // 3700) 769 / 732 / 752, of 384 961 / 931 / 960; even loads of 256 735 / 705 / 687; all rows in one expert, 8192 452 / 466 / 583,
    // 32768 685 / 694 / 1201.  (So the line could lie higher; it was drawn for the form of one block an expert.)
    const bool pieces = n_rows <= 256ll * num_experts;
    const int64_t chunks = xq_cdiv(n_rows, TN_CHUNK), parts = pieces ? num_experts + (chunks > 1 ? chunks - 1 : 0) : chunks;
    TnGroupedBatch b{};
    int32_t rfirst[kTnJobs];
    int nt = 1;
    int64_t blocks = 0, rblocks = 0;
    for (int i = 0; i < n; ++i) {
        const TnJob& j = jobs[i];
        const int64_t ldq = j.ldq > 0 ? j.ldq : j.r_pad;
        const int rc = tn_check(j.P, j.ldp, j.width, j.Q, ldq, j.r_pad, j.r_out);
        if (rc) return rc;
        if (j.width == 0 || j.r_out == 0) continue;
        const int k = b.n++;
        b.job[k] = TnArgs{j.P, j.ldp, j.width, j.Q, j.r_pad, j.r_out, n_rows, 0, j.transpose_out ? 1 : 0, j.out, offsets, nullptr, ldq, j.p_rows, j.out2, j.split_j};
        b.partial[k] = partial;
        b.col_tiles[k] = (int32_t)xq_cdiv(j.width, 128);
        b.first[k] = (int32_t)blocks;
        blocks += b.col_tiles[k] * parts;
        rfirst[k] = (int32_t)rblocks;
        rblocks += xq_cdiv(j.width * j.r_pad, 1024);
        if (j.r_pad > 32) nt = 2;
        partial += tn_partial_bytes(n_rows, j.width, j.r_pad) / 4;
    }
    if (b.n == 0) return XQ_OK;
    XQ_REQUIRE(blocks < (1ll << 31), "tn: %lld blocks", (long long)blocks);
    if (pieces) {
        if (nt == 1) tn_piece_kernel<1><<<(unsigned)blocks, 256, 0, stream>>>(b, num_experts);
        else tn_piece_kernel<2><<<(unsigned)blocks, 256, 0, stream>>>(b, num_experts);
    } else {
        if (nt == 1) tn_grouped_kernel<1><<<(unsigned)blocks, 256, 0, stream>>>(b, num_experts);
        else tn_grouped_kernel<2><<<(unsigned)blocks, 256, 0, stream>>>(b, num_experts);
    }
    XQ_CHECK_LAUNCH("tn(grouped)");
    if (pieces && chunks < 2) return XQ_OK;
    for (int k = 0; k < b.n; ++k) b.first[k] = rfirst[k];
    if (pieces) tn_grouped_reduce_kernel<true><<<dim3((unsigned)rblocks, (unsigned)(chunks - 1)), 256, 0, stream>>>(b, num_experts);
    else tn_grouped_reduce_kernel<false><<<dim3((unsigned)rblocks, (unsigned)num_experts), 256, 0, stream>>>(b, num_experts);
    XQ_CHECK_LAUNCH("tn(grouped reduce)");
    return XQ_OK;
}

int launch_tn(const bf16_t* P, int64_t ldp, int64_t width, const bf16_t* Q, int r_pad, int r_out, int64_t n_rows,
              bool transpose_out, float* out, float* partial, const int32_t* offsets, int32_t num_experts,
              hipStream_t stream, const int32_t* row_limit, int64_t ldq, const int32_t* p_rows) {
    const TnJob j{P, ldp, width, Q, ldq > 0 ? ldq : r_pad, r_pad, r_out, transpose_out, out, p_rows, nullptr, 0};
    if (!offsets) return launch_tn_multi(&j, 1, n_rows, partial, stream, row_limit);
    return launch_tn_grouped_multi(&j, 1, n_rows, partial, offsets, num_experts, stream);
}

}  // namespace xq
