// Low-rank (LoRA) helper kernels: factor preparation, the skinny "down"
// products (x.A^T, dy.B) and the weight-gradient products (dy^T.u, v^T.x).
// All are HBM-bound: they stream one large bf16 activation matrix once.
#pragma once

#include "xq_common.h"

namespace xq {

// The right-hand factor of a low-rank side term as the caller holds it: element (n, j), j < r, is f[n * ld + j], or f[j * ld + n]
// (transposed); columns from r to rp are zero.  With two factors (f[1] != NULL) the columns rp .. 2 rp are the second one's.
// The GEMM kernels round it to bf16 while they stage it: a dense call has no pass that prepares panels.
struct LowRankRight {
    const void* f[2];
    int64_t ld;
    int32_t r, rp;
    int32_t f32, transposed;
};
// 8 consecutive columns (chunk c) of row n, packed bf16; `which` >= 0 names the factor, < 0: by column.  Eight columns of a row are one
// or two 16-byte loads at whatever address they begin at, of a transposed factor eight loads in flight together: the branches on the
// type and the form lie around the loads and what is converted is kept as it came, since a branch between two loads makes the second
// wait for the first.
// A forward at r 64, us, element by element with a branch at each -> now: block-fp8 [5120, 448], 302 rows 16.0 -> 10.9 (gemm_mid_kernel), [1024,
// 320], 396 rows 13.0 -> 10.5 (128 x 128 tiles), [6272, 512], 2197 rows 32.3 -> 26.4 (gemm_dtl16_kernel); nf4 [7936, 2048], 1613 rows 68.7 ->
// 64.9 (gemm_dec_kernel); a third of that at r 32, nothing at r 8.
typedef u32x4 u32x4_any __attribute__((aligned(2)));
__device__ __forceinline__ u32x4 right_chunk(const LowRankRight& q, int which, int n, int c) {
    int j0 = c * 8, k = which;
    if (k < 0) {
        k = q.f[1] != nullptr && j0 >= q.rp ? 1 : 0;
        j0 -= k * q.rp;
    }
    const void* f = k ? q.f[1] : q.f[0];
    const int have = q.r - j0;                                         // columns of the chunk before the padding
    uint32_t raw[8];
    auto load = [&](auto T_) {
        typedef decltype(T_) T;
        if (q.transposed) {
            const T* p = (const T*)f + n;
#pragma unroll
            for (int e = 0; e < 8; ++e) raw[e] = p[(int64_t)(e < have ? j0 + e : q.r - 1) * q.ld];
        } else {
            const T* p = (const T*)f + (int64_t)n * q.ld;
            if (have >= 8) {
                const u32x4 lo = *(const u32x4_any*)(p + j0);
                u32x4 hi = {0u, 0u, 0u, 0u};
                if constexpr (sizeof(T) == 4) hi = *(const u32x4_any*)(p + j0 + 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) { raw[e] = lo[e]; raw[4 + e] = hi[e]; }
            } else {
                uint32_t v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = p[e < have ? j0 + e : q.r - 1];
#pragma unroll
                for (int e = 0; e < 8; ++e) raw[e] = sizeof(T) == 4 ? v[e] : e < 4 ? v[2 * (e & 3)] | v[2 * (e & 3) + 1] << 16 : 0u;
            }
        }
    };
    if (q.f32) load(uint32_t{});
    else load(uint16_t{});
    const bool pairs = !q.f32 && !q.transposed;                        // two bf16 to a word
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const uint32_t bits = q.f32 ? raw[e] : !pairs ? raw[e] << 16 : e & 1 ? raw[e >> 1] & 0xffff0000u : raw[e >> 1] << 16;
        v[e] = e < have ? __uint_as_float(bits) : 0.0f;
    }
    return u32x4{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
}

// the form a factor of a low-rank product comes in: [r, K] (rows along the contraction) or transposed, [K, r]
enum FactorMode { kFacBf16 = 0, kFacF32 = 1, kFacF32T = 2, kFacBf16T = 3 };
inline FactorMode factor_mode(int lora_dtype, bool transposed) {
    return lora_dtype == XQ_DT_F32 ? (transposed ? kFacF32T : kFacF32) : (transposed ? kFacBf16T : kFacBf16);
}

// T[rows, rp] = bf16(scale * In[rows, Kc] . F^T), dense rows, up to kLowRankJobs products in one launch.  nf = 2: a second
// factor of the same rank against the same rows, its result at T + t_step.  Ranks from r to rp come out zero.
constexpr int kLowRankJobs = 4;
struct LowRankJob {
    const bf16_t* In;
    int64_t ld_in, Kc;
    const void* F[2];
    int32_t nf, r, rp;
    float scale;
    bf16_t* T;
    int64_t ld_t, t_step;
};
int64_t lowrank_panel_bytes(int n, int64_t n_rows, int cols, int64_t Kc);   // scratch a launch of n products (nf * rp = cols each) may want
// scratch (may be NULL): memory for the fp32 sums of a contraction in splits, free again when the launch is done
int launch_lowrank(const LowRankJob* jobs, int n, int64_t n_rows, FactorMode mode, bf16_t* panels, hipStream_t stream, float* scratch = nullptr,
                   int64_t scratch_bytes = 0);

// Every LoRA panel of a call in one launch: job k converts a [n_src, R_in, C_in] fp32 / bf16 factor (n_src = 1 or
// the expert count) into bf16 [n_out, R_out, C_out], optionally transposed, zero padded; n_src == 1 < n_out repeats
// the one source matrix for every expert (a factor shared by all experts, handed to a kernel that indexes panels
// by expert).  `pitch` (0: C_out) is the row length of the destination, for a panel that is a column band of a
// wider one; `e_stride` (0: R_out * pitch) the distance between two experts' panels in the destination, for a panel
// that is a row band of a taller one.
constexpr int MAX_PANEL_JOBS = 6;
struct PanelJobs {
    const void* in[MAX_PANEL_JOBS];
    bf16_t* out[MAX_PANEL_JOBS];
    int64_t R_in[MAX_PANEL_JOBS], C_in[MAX_PANEL_JOBS], R_out[MAX_PANEL_JOBS], C_out[MAX_PANEL_JOBS], pitch[MAX_PANEL_JOBS];
    int64_t e_stride[MAX_PANEL_JOBS];
    int32_t n_src[MAX_PANEL_JOBS], n_out[MAX_PANEL_JOBS], transpose[MAX_PANEL_JOBS];
    int32_t in_f32, n;
    bf16_t* add(const void* src, int n_src_, int64_t r_in, int64_t c_in, bool tr, bf16_t* dst, int n_out_, int64_t r_out,
                int64_t c_out, int64_t pitch_ = 0, int64_t e_stride_ = 0) {
        in[n] = src; out[n] = dst; R_in[n] = r_in; C_in[n] = c_in; R_out[n] = r_out; C_out[n] = c_out;
        pitch[n] = pitch_ ? pitch_ : c_out;
        e_stride[n] = e_stride_ ? e_stride_ : r_out * pitch[n];
        n_src[n] = n_src_; n_out[n] = n_out_; transpose[n] = tr ? 1 : 0;
        ++n;
        return dst;
    }
};
int launch_panel_prep(const PanelJobs& jobs, hipStream_t stream);
int launch_factor_prep(const void* in, int in_dtype, int64_t R_in, int64_t C_in, bool transpose,
                       bf16_t* out, int64_t R_out, int64_t C_out, int64_t num_experts, hipStream_t stream);

// T[rows, r_pad] = bf16(scale * In[rows, Kc] . F[r_pad, Kc]^T), rows in expert order, F[e] = F + e*r_pad*Kc (or shared).
int launch_small_nt(const bf16_t* In, int64_t ld_in, int64_t n_rows, int64_t Kc, const bf16_t* F,
                    int r_pad, float scale, bf16_t* T, const int32_t* offsets,
                    const int32_t* tile_offsets, int32_t num_experts, bool shared_f, hipStream_t stream,
                    int64_t ld_t = 0,       // row pitch of T in elements (0: r_pad), to write a column band of a wider matrix
                    bf16_t* T2 = nullptr, int split = 0,    // result columns from `split` on go to T2 (same pitch): two panels' products from one pass
                    const int32_t* row_map = nullptr,       // grouped: product row i is made from row row_map[i] of In, and the
                    bf16_t* copy_out = nullptr, int64_t ld_copy = 0);   // gathered rows are also written to copy_out [rows, Kc] (if given)

// SwiGLU backward and the two low-rank products of its outputs in one pass (r_pad 16 or 32): dgate | dup as
// xq_silu_mul_bwd writes them, Tg = scale * dgate . Fg^T, Tu = scale * dup . Fu^T as two
// a low-rank launch on them would.  `partial`: silu_nt_partial_bytes() of scratch (dense; NULL keeps one block per 32 rows)
bool silu_bwd_nt_supported(int64_t cols, int r_pad);
int64_t silu_nt_partial_bytes(int64_t n_rows, int64_t cols, int r_pad);
int launch_silu_bwd_nt(const bf16_t* gate, const bf16_t* up, int64_t ld_gu, const bf16_t* dh, int64_t ld_dh, bf16_t* dgate,
                       bf16_t* dup, int64_t ld_out, int64_t n_rows, int64_t cols, const void* Fg, const void* Fu, FactorMode mode, int r, int r_pad,
                       float scale, bf16_t* Tg, bf16_t* Tu, int64_t ld_t, float* partial, hipStream_t stream,
                       // routed rows in expert order (offsets != NULL): a factor pair per expert ([E][r_pad][cols]) unless
                       // shared, the rows' routing weights applied and (d_row_w != NULL) their gradients written
                       const int32_t* offsets = nullptr, const int32_t* tile_offsets = nullptr, int32_t num_experts = 1,
                       bool shared_fg = true, bool shared_fu = true, const float* row_w = nullptr, float* d_row_w = nullptr,
                       float swiglu_limit = 0.0f);     // > 0: the gate pre-activation is clamped to [-limit, limit], its gradient masked outside

// the forward in the same organisation: h = SwiGLU(gate, up) (routed rows: times the row's weight), T = scale * h . F^T, F as
// bf16 panels; dense rows in blocks of 32 over all columns, for launches that fill the chip so
int launch_silu_fwd_nt(const bf16_t* gate, const bf16_t* up, int64_t ld_gu, bf16_t* h, int64_t ld_h, int64_t n_rows, int64_t cols,
                       const bf16_t* F, int r_pad, float scale, bf16_t* T, int64_t ld_t, hipStream_t stream, const int32_t* offsets = nullptr,
                       const int32_t* tile_offsets = nullptr, int32_t num_experts = 1, bool shared_f = true, const float* row_w = nullptr,
                       float swiglu_limit = 0.0f);

// xq_silu_mul_fwd / xq_silu_mul_bwd with a SwiGLU limit on the gate pre-activation (ops/moe/triton.py:127-141; <= 0: none)
int silu_mul_fwd_limit(const void* gate, const void* up, int64_t ld_in, const float* row_w, void* h, int64_t ld_h, int64_t rows,
                       int64_t cols, float limit, void* stream);
int silu_mul_bwd_limit(const void* gate, const void* up, int64_t ld_in, const void* dh, int64_t ld_dh, const float* row_w, void* dgate,
                       void* dup, int64_t ld_out, float* d_row_w, int64_t rows, int64_t cols, float limit, void* stream);

// out[c][j] (or out[j][c] when transpose_out) = sum_m P[m][c] * Q[m][j], fp32.
//   dense: all rows, split over `splits` row ranges, partials in `partial`
//          ([splits][width][r_pad] fp32) reduced in fixed order (deterministic);
//   grouped: out[e] over rows [offsets[e], offsets[e+1]); zero for empty experts.
// r_out is the number of valid columns of Q (<= r_pad) written.
// Dense products of the same rows can share a launch (launch_tn_multi): their partials lie one after the other,
// tn_partial_bytes() each.  out2 (may be NULL): columns of Q from split_j on are a second result's columns.
constexpr int kTnJobs = 6;
struct TnJob {
    const bf16_t* P;
    int64_t ldp, width;
    const bf16_t* Q;
    int64_t ldq;
    int32_t r_pad, r_out;
    bool transpose_out;
    float* out;
    const int32_t* p_rows;
    float* out2;
    int32_t split_j;
};
int launch_tn_multi(const TnJob* jobs, int n, int64_t n_rows, float* partial, hipStream_t stream, const int32_t* row_limit = nullptr);
// ... and so can grouped ones (one set of offsets)
int launch_tn_grouped_multi(const TnJob* jobs, int n, int64_t n_rows, float* partial, const int32_t* offsets, int32_t num_experts,
                            hipStream_t stream);
int64_t tn_partial_bytes(int64_t n_rows, int64_t width, int r_pad);
int launch_tn(const bf16_t* P, int64_t ldp, int64_t width, const bf16_t* Q, int r_pad, int r_out,
              int64_t n_rows, bool transpose_out, float* out, float* partial,
              const int32_t* offsets, int32_t num_experts, hipStream_t stream,
              const int32_t* row_limit = nullptr,    // dense form: contract only rows below *row_limit (device value)
              int64_t ldq = 0,                       // row pitch of Q in elements (0: r_pad), for a column band of a wider matrix
              const int32_t* p_rows = nullptr);      // optional: row m of the contraction is row p_rows[m] of P (Q rows stay in order)

int launch_zero_fill(void* p, int64_t bytes, hipStream_t stream);

// What a product's fp32 sums have to equal.  any: the kernels are free to sum in the order that suits the sizes.  kept: the order of the
// kernel that the sizes choose among gemm_256_kernel, gemm_mid_kernel, gemm_dec_kernel and gemm_dtl16_kernel (expert banks: 256 x 256 tiles of
// block-fp8 in gemm_dtl16_kernel's order, everything else in gemm_256_kernel's).  A bf16
// rounding of such a sum that flips with the order moves what is computed from it by some 2e-4 (2-norm), in fp32 results too: that is many times
// fp32's rounding.  So the products that fp32 gradients are computed from, or that one program runs in more than one form, are kept.
enum class SumOrder { any, kept };
// fused dequant-GEMM launcher (xq_gemm.hip).  `two`: a grouped launch over two block-fp8 banks of one shape -- the
// forward (contract_cols false) writes [rows, 2 * cols] with the second bank's columns, side term su2 / lora_right2,
// after the first's; the dgrad (contract_cols true) contracts A [rows, 2 * cols] against both banks into one sum.
struct TwoBanks {
    const xq_weight* w2;
    const bf16_t* su2;
    const bf16_t* lora_right2;
    int32_t a_off2;              // 4-bit dgrad: the second bank's activations lie that many columns further right
};
int64_t tile_gemm_split_bytes(int64_t n_rows, int64_t Nout, int64_t Kc);     // split-K scratch a dense launch may want
int64_t tile_gemm_partial_bytes(int fmt, int64_t n_rows, int64_t Nout, int64_t Kc);   // ... or the decoded image of a weight of that format (< 0: of any)
bool two_banks_supported(const xq_weight* w);
bool banks_side_by_side(const xq_weight* a, const xq_weight* b, bool contract_cols, int64_t n_rows, SumOrder order);
bool two_dense_supported(const xq_weight* w);   // dense [N, K] pair: one dgrad launch, dX = [dY1 | dY2] . [W1 ; W2]
int launch_gate_up_swiglu(const xq_weight* wg, const xq_weight* wu, const bf16_t* x, int64_t ldx, int64_t M,
                          const bf16_t* su_g, const bf16_t* su_u, int64_t ld_su, const LowRankRight& right,
                          int r_pad, const bf16_t* bias_g, const bf16_t* bias_u, bf16_t* gu, int64_t ldgu, bf16_t* h,
                          int64_t ldh, hipStream_t stream);
bool gate_up_side_by_side(const xq_weight* wg, const xq_weight* wu, const bf16_t* x, int64_t ldx, int64_t M, const bf16_t* bias_g,
                          const bf16_t* bias_u, const bf16_t* gu, int64_t ldgu);
int launch_gate_up(const xq_weight* wg, const xq_weight* wu, const bf16_t* x, int64_t ldx, int64_t M, const bf16_t* su_g, const bf16_t* su_u,
                   int64_t ld_su, const LowRankRight& right, int r_pad, const bf16_t* bias_g, const bf16_t* bias_u, bf16_t* gu, int64_t ldgu,
                   hipStream_t stream, const char* who);
int launch_tile_gemm(const xq_weight* w, bool contract_cols, const bf16_t* A, int64_t lda, int64_t n_rows,
                     const int32_t* offsets, const int32_t* tile_offsets, const bf16_t* su, const bf16_t* lora_right,
                     int r_pad, const bf16_t* bias, bf16_t* C, int64_t ldc, hipStream_t stream, const char* who,
                     float* partial, int64_t partial_bytes, const TwoBanks* two = nullptr,
                     const LowRankRight* right = nullptr,   // dense: the side term's right-hand factor (then lora_right is NULL)
                     SumOrder order = SumOrder::any,
                     const int32_t* a_rows = nullptr,    // grouped, optional: row i of the problem is row a_rows[i] of A,
                     int64_t a_span_rows = 0);           // ... which has this many rows (0: not known)
bool tile_gemm_takes_row_map(const xq_weight* w);        // ... which only the pipelined tile kernel does

int num_cus();   // compute units of the current device (xq_gemm.hip)

// skinny-M (M <= 64) forward path, xq_skinny.hip
bool skinny_supported(const xq_weight* w, int64_t M);
int64_t skinny_workspace_bytes(int64_t M, int64_t N, int64_t K, int r_pad);
int launch_skinny(const xq_weight* w, const bf16_t* x, int64_t ldx, int64_t M, const void* lora_A, const void* lora_B,
                  int lora_dtype, int r, float scaling, const bf16_t* bias, bf16_t* y, int64_t ldy, void* workspace,
                  int64_t workspace_bytes, hipStream_t stream);

}  // namespace xq
