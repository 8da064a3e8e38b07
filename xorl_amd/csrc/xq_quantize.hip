// Encoding a weight: bf16 / fp32 values -> packed codes and scales, in the reference quantizers' arithmetic bit for bit:
//   int4   scale = max(amax, 1e-12) * 2/15, code = trunc(x / scale + 8.5)      ops/quantize/int4_quantize.py:12-41
//          (bf16 scales: the symmetric rule scale = bf16(amax / 7), code = rne(x / scale) + 8; not in the reference)
//   nvfp4  code = e2m1(x * (6 / amax)), scale = e4m3(amax / tensor amax * 448)  ops/quantize/nvfp4_quantize.py:25-60
//   nf4    code = nearest level of x * (1 / amax)                               ops/quantize/nf4_quantize.py:20-56
//   fp8    s = max(amax / 448, 1e-12) per 128 x 128 tile, e4m3(x / s)           ops/quantize/block_fp8_gkn_quantize.py:40-121
//
// Bound by HBM: the weight is read once (16-byte loads, held in registers between the group's absmax and its codes) and the
// codes are written once.  A NaN stays visible: it makes its group's scale NaN (and nvfp4's global scale), and an infinity gives
// an infinite scale, as in the torch forms.  Written in torch operations the same arithmetic was 15-25 passes over fp32 copies of the weight:
// [12288, 4096] bf16 -> nvfp4 took 2250 us where the bytes need 26 at a large copy's rate.
#include "xq_common.h"
#include "xq_codes.h"

namespace xq {
namespace {

constexpr int kMaxBlocks = 2048;    // of the grid-stride kernels: the partial maxima of a launch are read whole by the next one

struct QuantArgs {
    const void* x;
    int64_t rows, cols;
    int32_t group;
    bool sym;                   // int4: bf16 scales, symmetric rule
    float amax_scale;           // fp8
    const float* gamax;         // nvfp4: the tensor amax where the caller knows it
    uint8_t* codes;
    void* scales;
    float* gscale;              // nvfp4: one float
    void* amax_out;             // nvfp4 without a known tensor amax: the blocks' amax, in x's type (it is one of x's values),
    float* partial;             // and each thread block's maximum over them, for nvfp4_scales_kernel
};

// the larger / the smaller of the two, NaN where either is (fmaxf and fminf return the other operand); one instruction
__device__ __forceinline__ float max_nan(float a, float b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ float min_nan(float a, float b) { return __builtin_elementwise_minimum(a, b); }
// into [-top, top], NaN kept
__device__ __forceinline__ float clamp_nan(float v, float top) { return max_nan(min_nan(v, top), -top); }

__device__ __forceinline__ void unpack8(u32x4 w, float* v) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = __uint_as_float(w[i] << 16);
        v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
}

// 8 values of x from element `at`
template <bool F32>
struct Raw8 {
    u32x4 w[F32 ? 2 : 1];
    __device__ __forceinline__ void load(const void* x, int64_t at) {
        if constexpr (F32) {
            w[0] = *(const u32x4*)((const float*)x + at);
            w[1] = *(const u32x4*)((const float*)x + at + 4);
        } else {
            w[0] = *(const u32x4*)((const bf16_t*)x + at);
        }
    }
    __device__ __forceinline__ void get(float* v) const {
        if constexpr (F32) {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = __uint_as_float(w[i >> 2][i & 3]);
        } else {
            unpack8(w[0], v);
        }
    }
};

// what a group's absmax makes of its values
template <int FMT>
struct GroupRule {
    float mul, scale;
    bool sym;
    const Nf4Bucket* nf4;
    __device__ __forceinline__ GroupRule(float amax, bool sym_, const Nf4Bucket* t) : sym(sym_), nf4(t) {
        if constexpr (FMT == XQ_FMT_NVFP4) {
            scale = max_nan(amax, 1e-12f);
            mul = 4.0f * (6.0f / scale);                 // fp4_code4 takes 4 x the scaled value
        } else if constexpr (FMT == XQ_FMT_NF4) {
            scale = max_nan(amax, 1e-12f);
            mul = 1.0f / scale;
        } else if (sym) {
            scale = round_bf16(amax / 7.0f);
            mul = scale > 0.0f ? 1.0f / scale : 0.0f;
        } else {
            scale = max_nan(amax, 1e-12f) * (float)(2.0 / 15.0);
            mul = 1.0f / scale;
        }
    }
    __device__ __forceinline__ uint32_t code(float x) const {
        if constexpr (FMT == XQ_FMT_NVFP4) {
            return fp4_code4(x * mul);
        } else if constexpr (FMT == XQ_FMT_NF4) {
            return nf4_code(__builtin_amdgcn_fmed3f(x * mul, -1.0f, 1.0f), nf4);      // (NaN: -1, code 0)
        } else {
            if (sym) {
                // x / scale rounded to fp32, as one multiplication by the rounded reciprocal and one correction: the remainder is
                // exact, and with a bf16 scale no quotient lies closer than 2^-9 ulp to a rounding boundary, far outside the
                // correction's error.  (Tiny scales, whose remainders would be denormal, take the division; zero, infinite and NaN scales code 8.)
                // [12288, 4096]: 44 -> 30 us
                float q = x * mul;
                q = __builtin_fmaf(__builtin_fmaf(-q, scale, x), mul, q);
                if (!(scale >= 0x1p-60f && scale < INFINITY)) q = scale > 0.0f && scale < INFINITY ? x / scale : 0.0f;
                return (uint32_t)((int)__builtin_amdgcn_fmed3f(__builtin_rintf(q), -7.0f, 7.0f) + 8);
            }
            return (uint32_t)__builtin_amdgcn_fmed3f(__fadd_rn(__fmul_rn(x, mul), 8.5f), 0.0f, 15.0f);      // (NaN: 0)
        }
    }
};

__device__ __forceinline__ uint8_t nvfp4_block_scale(float amax, float gamax) {
    const float bs = clamp_nan(amax / gamax * 448.0f, 448.0f);
    return (uint8_t)(__builtin_amdgcn_cvt_pk_fp8_f32(bs, 0.0f, 0u, false) & 0xffu);
}

__device__ __forceinline__ float nvfp4_global_scale(float gamax) { return gamax * (1.0f / 6.0f) / 448.0f; }

// this block's maximum of `m` over its threads -> partial[blockIdx.x]
__device__ __forceinline__ void store_block_max(float m, float* partial) {
    __shared__ float wm[4];
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) m = max_nan(m, __shfl_xor(m, d, 64));
    if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = max_nan(max_nan(wm[0], wm[1]), max_nan(wm[2], wm[3]));
}

template <bool F32>
__device__ __forceinline__ void store_amax(void* out, int64_t i, float m) {
    if constexpr (F32) ((float*)out)[i] = m;
    else ((bf16_t*)out)[i] = (bf16_t)(__float_as_uint(m) >> 16);         // |x| of a bf16 value: exact
}

// groups along the fast axis: a thread takes 16 consecutive values, group / 16 neighbouring lanes (a power of two) a group
template <int FMT, bool F32>
__global__ void __launch_bounds__(256) quant_flat_kernel(QuantArgs g, int64_t runs) {
    __shared__ Nf4Bucket nf4[FMT == XQ_FMT_NF4 ? 32 : 1];
    if (FMT == XQ_FMT_NF4) {
        if (threadIdx.x < 32) nf4[threadIdx.x] = nf4_bucket(threadIdx.x);
        __syncthreads();
    }
    const int lanes = g.group >> 4;
    const float gm = FMT == XQ_FMT_NVFP4 && g.gamax ? max_nan(g.gamax[0], 1e-12f) : 1.0f;
    float top = 0.0f;
    // (the lanes of a group are in range together: the element count is a multiple of the group)
    for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < runs; t += (int64_t)gridDim.x * 256) {
        Raw8<F32> a, b;
        a.load(g.x, t * 16);
        b.load(g.x, t * 16 + 8);
        float v[16];
        a.get(v);
        b.get(v + 8);
        float m = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) m = max_nan(m, fabsf(v[i]));
        for (int d = 1; d < lanes; d <<= 1) m = max_nan(m, __shfl_xor(m, d, 64));
        const GroupRule<FMT> rule(m, g.sym, nf4);
        uint32_t w[2] = {0u, 0u};
#pragma unroll
        for (int i = 0; i < 16; ++i) w[i >> 3] |= rule.code(v[i]) << (4 * (i & 7));
        *(u32x2*)(g.codes + t * 8) = u32x2{w[0], w[1]};
        if constexpr (FMT == XQ_FMT_NVFP4) {
            if (g.gamax) ((uint8_t*)g.scales)[t] = nvfp4_block_scale(rule.scale, gm);
            else store_amax<F32>(g.amax_out, t, m);
            top = max_nan(top, m);
        } else if ((threadIdx.x & (lanes - 1)) == 0) {
            if (FMT == XQ_FMT_INT4 && g.sym) ((bf16_t*)g.scales)[t / lanes] = to_bf16(rule.scale);
            else ((float*)g.scales)[t / lanes] = rule.scale;
        }
    }
    if constexpr (FMT == XQ_FMT_NVFP4) {
        if (!g.gamax) store_block_max(top, g.partial);
        else if (blockIdx.x == 0 && threadIdx.x == 0) g.gscale[0] = nvfp4_global_scale(gm);
    }
}

// groups of 16, 32 or 64 down the rows of [rows, cols], pairs of rows in a byte: a wave takes 64 rows x 128 columns, a lane
// 16 rows of 8 columns (16 lanes make a row's 256 bytes; the lanes 16 and 32 further hold the next 16 rows of the same
// columns, and a group of 32 or 64 rows meets over them)
template <int FMT, bool F32>
__global__ void __launch_bounds__(256) quant_gkn_kernel(QuantArgs g, int64_t col_blocks, int64_t waves) {
    __shared__ Nf4Bucket nf4[FMT == XQ_FMT_NF4 ? 32 : 1];
    if (FMT == XQ_FMT_NF4) {
        if (threadIdx.x < 32) nf4[threadIdx.x] = nf4_bucket(threadIdx.x);
        __syncthreads();
    }
    const int lane = threadIdx.x & 63, rq = lane >> 4, cq = lane & 15;
    const float gm = FMT == XQ_FMT_NVFP4 && g.gamax ? max_nan(g.gamax[0], 1e-12f) : 1.0f;
    float top = 0.0f;
    for (int64_t wv = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); wv < waves; wv += (int64_t)gridDim.x * 4) {
        const int64_t rb = wv / col_blocks, cb = wv - rb * col_blocks;
        const int64_t row = rb * 64 + rq * 16, col = cb * 128 + cq * 8;
        const bool ok = row < g.rows && col < g.cols;             // rows % group == 0, cols % 8 == 0: whole pieces
        const int64_t lr = row < g.rows ? row : g.rows - 16, lc = col < g.cols ? col : g.cols - 8;
        Raw8<F32> raw[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) raw[i].load(g.x, (lr + i) * g.cols + lc);
        float m[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            float v[8];
            raw[i].get(v);
#pragma unroll
            for (int c = 0; c < 8; ++c) m[c] = max_nan(m[c], fabsf(v[c]));
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            if (g.group >= 32) m[c] = max_nan(m[c], __shfl_xor(m[c], 16, 64));
            if (g.group >= 64) m[c] = max_nan(m[c], __shfl_xor(m[c], 32, 64));
        }
        uint32_t w[8][2];
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i][0] = w[i][1] = 0u;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const GroupRule<FMT> rule(m[c], g.sym, nf4);
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                float v[8];
                raw[i].get(v);
                w[i >> 1][c >> 2] |= rule.code(v[c]) << (8 * (c & 3) + 4 * (i & 1));
            }
            if (ok && (row & (g.group - 1)) == 0) {
                const int64_t si = row / g.group * g.cols + col + c;
                if constexpr (FMT == XQ_FMT_NVFP4) {
                    if (g.gamax) ((uint8_t*)g.scales)[si] = nvfp4_block_scale(rule.scale, gm);
                    else store_amax<F32>(g.amax_out, si, m[c]);
                } else if (FMT == XQ_FMT_INT4 && g.sym) {
                    ((bf16_t*)g.scales)[si] = to_bf16(rule.scale);
                } else {
                    ((float*)g.scales)[si] = rule.scale;
                }
            }
            top = max_nan(top, ok ? m[c] : 0.0f);
        }
        if (ok) {
#pragma unroll
            for (int i = 0; i < 8; ++i) *(u32x2*)(g.codes + (row / 2 + i) * g.cols + col) = u32x2{w[i][0], w[i][1]};
        }
    }
    if constexpr (FMT == XQ_FMT_NVFP4) {
        if (!g.gamax) store_block_max(top, g.partial);
        else if (blockIdx.x == 0 && threadIdx.x == 0) g.gscale[0] = nvfp4_global_scale(gm);
    }
}

// nvfp4 without a known tensor amax, second launch: the tensor amax from the first launch's partial maxima (every block
// reduces them: at most 8 KB from L2), then the block scales, four a thread
template <bool F32>
__global__ void __launch_bounds__(256) nvfp4_scales_kernel(const void* amax, int64_t n, const float* partial, int parts, uint8_t* scales, float* gscale) {
    __shared__ float wm[4];
    float m = 0.0f;
    for (int i = threadIdx.x; i < parts; i += 256) m = max_nan(m, partial[i]);
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) m = max_nan(m, __shfl_xor(m, d, 64));
    if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
    __syncthreads();
    const float gm = max_nan(max_nan(max_nan(wm[0], wm[1]), max_nan(wm[2], wm[3])), 1e-12f);
    if (blockIdx.x == 0 && threadIdx.x == 0) gscale[0] = nvfp4_global_scale(gm);
    for (int64_t t = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4; t < n; t += (int64_t)gridDim.x * 1024) {
        float a[4];
        if (t + 4 <= n) {
            if constexpr (F32) {
                const f32x4 v = *(const f32x4*)((const float*)amax + t);
                for (int i = 0; i < 4; ++i) a[i] = v[i];
            } else {
                const u32x2 v = *(const u32x2*)((const bf16_t*)amax + t);
                a[0] = __uint_as_float(v[0] << 16); a[1] = __uint_as_float(v[0] & 0xffff0000u);
                a[2] = __uint_as_float(v[1] << 16); a[3] = __uint_as_float(v[1] & 0xffff0000u);
            }
            uint32_t w = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) w |= (uint32_t)nvfp4_block_scale(max_nan(a[i], 1e-12f), gm) << (8 * i);
            *(uint32_t*)(scales + t) = w;
        } else {
            for (int64_t i = t; i < n; ++i)
                scales[i] = nvfp4_block_scale(max_nan(F32 ? ((const float*)amax)[i] : bf16_to_f32(((const bf16_t*)amax)[i]), 1e-12f), gm);
        }
    }
}

// block-fp8: a thread block takes one 128 x 128 tile (partial at the edges), a thread 8 rows of 8 columns
template <bool F32>
__global__ void __launch_bounds__(256) quant_fp8_kernel(QuantArgs g) {
    __shared__ float wm[4];
    const int tid = threadIdx.x;
    const int64_t r0 = (int64_t)blockIdx.y * 128 + (tid >> 4), col = (int64_t)blockIdx.x * 128 + (tid & 15) * 8;
    const int64_t lc = col < g.cols ? col : g.cols - 8;           // cols % 8 == 0
    Raw8<F32> raw[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int64_t row = r0 + 16 * i;
        raw[i].load(g.x, (row < g.rows ? row : g.rows - 1) * g.cols + lc);      // clamped into the tile's own edge: the maximum is unchanged
    }
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        float v[8];
        raw[i].get(v);
#pragma unroll
        for (int c = 0; c < 8; ++c) m = max_nan(m, fabsf(v[c]));
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) m = max_nan(m, __shfl_xor(m, d, 64));
    if ((tid & 63) == 0) wm[tid >> 6] = m;
    __syncthreads();
    m = max_nan(max_nan(wm[0], wm[1]), max_nan(wm[2], wm[3]));
    const float s = max_nan(m * g.amax_scale / 448.0f, 1e-12f);
    if (tid == 0) ((float*)g.scales)[(int64_t)blockIdx.y * gridDim.x + blockIdx.x] = s;
    if (col >= g.cols) return;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int64_t row = r0 + 16 * i;
        if (row >= g.rows) break;
        float v[8];
        raw[i].get(v);
#pragma unroll
        for (int c = 0; c < 8; ++c) v[c] = clamp_nan(v[c] / s, 448.0f);
        uint32_t w[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            w[h] = __builtin_amdgcn_cvt_pk_fp8_f32(v[4 * h], v[4 * h + 1], 0u, false);
            w[h] = __builtin_amdgcn_cvt_pk_fp8_f32(v[4 * h + 2], v[4 * h + 3], w[h], true);
        }
        *(u32x2*)(g.codes + row * g.cols + col) = u32x2{w[0], w[1]};
    }
}

template <int FMT>
void launch_4bit(const QuantArgs& g, bool f32, bool gkn, int64_t runs, int64_t col_blocks, int64_t waves, unsigned grid, hipStream_t s) {
    if (gkn) {
        if (f32) quant_gkn_kernel<FMT, true><<<grid, 256, 0, s>>>(g, col_blocks, waves);
        else quant_gkn_kernel<FMT, false><<<grid, 256, 0, s>>>(g, col_blocks, waves);
    } else {
        if (f32) quant_flat_kernel<FMT, true><<<grid, 256, 0, s>>>(g, runs);
        else quant_flat_kernel<FMT, false><<<grid, 256, 0, s>>>(g, runs);
    }
}

}  // namespace
}  // namespace xq

using namespace xq;

extern "C" int64_t xq_quantize_workspace_bytes(int format, int64_t rows, int64_t cols) {
    return format == XQ_FMT_NVFP4 && rows > 0 && cols > 0 ? rows * cols / 16 * 4 + kMaxBlocks * 4 + 512 : 0;
}

extern "C" int xq_quantize(int format, int layout, const void* x, int x_dtype, int64_t rows, int64_t cols, int32_t group, float amax_scale,
                           const float* global_amax, void* codes, void* scales, int scale_dtype, float* global_scale, void* workspace,
                           int64_t workspace_bytes, void* stream_) {
    static const char* who = "xq_quantize";
    XQ_REQUIRE(format == XQ_FMT_INT4 || format == XQ_FMT_NVFP4 || format == XQ_FMT_FP8 || format == XQ_FMT_NF4, "%s: bad format %d", who, format);
    XQ_REQUIRE(layout == XQ_LAYOUT_FLAT || layout == XQ_LAYOUT_GKN, "%s: bad layout %d", who, layout);
    XQ_REQUIRE(x_dtype == XQ_DT_BF16 || x_dtype == XQ_DT_F32, "%s: values are bf16 or fp32", who);
    XQ_REQUIRE(rows >= 1 && cols >= 1 && rows < (1ll << 31) && cols < (1ll << 40) && rows * cols < (1ll << 42), "%s: bad shape [%lld, %lld]", who, (long long)rows, (long long)cols);
    XQ_REQUIRE(x && codes && scales && xq_aligned(x, 16) && xq_aligned(codes, 8), "%s: values 16-byte and codes 8-byte aligned, neither NULL", who);
    hipStream_t stream = (hipStream_t)stream_;
    const bool f32 = x_dtype == XQ_DT_F32;
    QuantArgs g{};
    g.x = x; g.rows = rows; g.cols = cols; g.group = group; g.codes = (uint8_t*)codes; g.scales = scales; g.amax_scale = amax_scale;
    if (format == XQ_FMT_FP8) {
        XQ_REQUIRE(group == 128 && cols % 8 == 0 && scale_dtype == XQ_SCALE_F32 && amax_scale > 0.0f, "%s: block-fp8 takes 128 x 128 blocks, columns in multiples of 8 and fp32 scales", who);
        const dim3 grid((unsigned)xq_cdiv(cols, 128), (unsigned)xq_cdiv(rows, 128));
        XQ_REQUIRE(grid.y < 65536, "%s: too many rows", who);
        if (f32) quant_fp8_kernel<true><<<grid, 256, 0, stream>>>(g);
        else quant_fp8_kernel<false><<<grid, 256, 0, stream>>>(g);
        XQ_CHECK_LAUNCH(who);
        return XQ_OK;
    }
    const bool gkn = layout == XQ_LAYOUT_GKN;
    XQ_REQUIRE(group >= 16 && (group & (group - 1)) == 0 && group <= (gkn ? 64 : 1024), "%s: groups of 16 .. %d, a power of two; got %d", who, gkn ? 64 : 1024, group);
    XQ_REQUIRE((gkn ? rows % group : rows * cols % group) == 0, "%s: the group %d does not divide the grouped extent", who, group);
    XQ_REQUIRE(!gkn || cols % 8 == 0, "%s: columns in multiples of 8", who);
    XQ_REQUIRE(format != XQ_FMT_NVFP4 || (group == 16 && scale_dtype == XQ_SCALE_E4M3 && global_scale), "%s: nvfp4 takes blocks of 16, e4m3 scales and a global scale output", who);
    XQ_REQUIRE(format != XQ_FMT_NF4 || scale_dtype == XQ_SCALE_F32, "%s: nf4 scales are fp32", who);
    XQ_REQUIRE(format != XQ_FMT_INT4 || scale_dtype == XQ_SCALE_F32 || scale_dtype == XQ_SCALE_BF16, "%s: int4 scales are fp32 or bf16", who);
    g.sym = format == XQ_FMT_INT4 && scale_dtype == XQ_SCALE_BF16;
    const int64_t runs = rows * cols / 16, col_blocks = xq_cdiv(cols, 128), waves = xq_cdiv(rows, 64) * col_blocks;
    const int64_t want = gkn ? xq_cdiv(waves, 4) : xq_cdiv(runs, 256);
    const unsigned grid = (unsigned)(want < kMaxBlocks ? want : kMaxBlocks);
    if (format == XQ_FMT_NVFP4) {
        g.gamax = global_amax;
        g.gscale = global_scale;
        if (!global_amax) {
            XQ_REQUIRE(workspace && xq_aligned(workspace, 256) && workspace_bytes >= xq_quantize_workspace_bytes(format, rows, cols),
                       "%s: workspace missing, misaligned or smaller than xq_quantize_workspace_bytes()", who);
            XQ_REQUIRE(xq_aligned(scales, 4), "%s: scales must be 4-byte aligned", who);
            g.partial = (float*)workspace;
            g.amax_out = (uint8_t*)workspace + kMaxBlocks * 4;
        }
        launch_4bit<XQ_FMT_NVFP4>(g, f32, gkn, runs, col_blocks, waves, grid, stream);
        XQ_CHECK_LAUNCH(who);
        if (!global_amax) {
            const int64_t sb = xq_cdiv(runs, 1024);
            const unsigned sgrid = (unsigned)(sb < kMaxBlocks ? sb : kMaxBlocks);
            if (f32) nvfp4_scales_kernel<true><<<sgrid, 256, 0, stream>>>(g.amax_out, runs, g.partial, (int)grid, (uint8_t*)scales, global_scale);
            else nvfp4_scales_kernel<false><<<sgrid, 256, 0, stream>>>(g.amax_out, runs, g.partial, (int)grid, (uint8_t*)scales, global_scale);
            XQ_CHECK_LAUNCH(who);
        }
        return XQ_OK;
    }
    if (format == XQ_FMT_NF4) launch_4bit<XQ_FMT_NF4>(g, f32, gkn, runs, col_blocks, waves, grid, stream);
    else launch_4bit<XQ_FMT_INT4>(g, f32, gkn, runs, col_blocks, waves, grid, stream);
    XQ_CHECK_LAUNCH(who);
    return XQ_OK;
}
