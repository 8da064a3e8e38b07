// xq_mlp_fwd / xq_mlp_bwd: the dense SwiGLU MLP of three QLoRA linears (gate, up, down) as two calls.
// Host code only.  The program is the reference's Qwen3MLP.forward over three QLoRALinear modules
// (models/transformers/qwen3/modeling_qwen3.py:60-81 with qlora/modules/linear.py:369-385 and
// ops/fused_silu_and_mul.py:22-60) and its backward, composed from this library's kernels on the caller's stream
// so that work the three separate module calls repeat is shared:
//   forward   one pass over x gives both low-rank intermediates; block-fp8 gate / up run as one launch whose
//             epilogue also writes h = bf16(silu(gate)) * up, or as one launch of plain tiles where that fills the chip better
//             than two;
//   backward  the dgrads of gate and up are one launch, dX = [dgate | dup] . [Wg ; Wu] + [v_g | v_u] . [A_g ; A_u],
//             and the two A gradients come from one pass over x.
// Other formats (and shapes the fused forms do not take) run the same program launch by launch.
#include "xq_lora.h"
#include "xq_skinny.h"
#include <algorithm>
#include <atomic>
#include <stdlib.h>

namespace xq {
namespace {

inline int64_t al256(int64_t b) { return (b + 255) & ~(int64_t)255; }
inline int r_pad_of(int r) { return r <= 0 ? 0 : ((r + 15) / 16) * 16; }

struct Carve {
    uint8_t* base;
    int64_t used;
    template <typename T>
    T* take(int64_t bytes) {
        T* p = (T*)(base + used);
        used += al256(bytes);
        return p;
    }
};

struct Dims {
    int64_t M, H, I;
    int r, rp;
};

// a[m][c] = bf16(a[m][c] + b[m][c]): the two shares of dX when the dgrads of gate and up run as separate launches
__global__ void __launch_bounds__(256) add_rows_kernel(bf16_t* a, int64_t lda, const bf16_t* b, int64_t ldb, int64_t rows, int64_t cols8) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= rows * cols8) return;
    const int64_t m = t / cols8, c = (t - m * cols8) * 8;
    u32x4 av = *(const u32x4*)(a + m * lda + c), bv = *(const u32x4*)(b + m * ldb + c), o;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        o[i] = pack_bf16x2(bf16_to_f32((bf16_t)(av[i] & 0xffffu)) + bf16_to_f32((bf16_t)(bv[i] & 0xffffu)),
                           bf16_to_f32((bf16_t)(av[i] >> 16)) + bf16_to_f32((bf16_t)(bv[i] >> 16)));
    *(u32x4*)(a + m * lda + c) = o;
}

// gate and up of a block-fp8 MLP as ONE launch with the SwiGLU in its epilogue (1), or as two launches followed by the pass
// that writes h and forms s * h . A_d^T on the way (0, the default: the two plain launches run at a higher rate than the
// launch with the wide epilogue, and the step is level or slightly shorter).  XQ_MLP_GU in the environment sets it at load
// time, xq_set_mlp_gate_up_fused() at run time.  It is only the default of a forward: xq_mlp_saved::gate_up_fused carries the
// form a forward used (or was asked for) to its backward, which lays out the saved low-rank intermediates by that field.
static std::atomic<int> g_mlp_gu{[] { const char* e = getenv("XQ_MLP_GU"); return e ? atoi(e) : 0; }()};
// XQ_MLP_SILU_NT=0: the SwiGLU backward and the two low-rank products of its outputs as three launches (A/B measurements;
// same bits either way)
static const int g_mlp_silu_nt = [] { const char* e = getenv("XQ_MLP_SILU_NT"); return e ? atoi(e) : 1; }();
// `asked`: xq_mlp_saved::gate_up_fused on entry to the forward (< 0: the process-wide default decides)
bool fuse_gate_up_fwd(const xq_weight* gate, const xq_weight* up, int asked) {
    return (asked < 0 ? g_mlp_gu.load() != 0 : asked != 0) && gate->format == XQ_FMT_FP8 && up->format == XQ_FMT_FP8;
}

// Where the two low-rank intermediates lie in su_gate_up (M * 2 * rp elements): as the column bands [0, rp) and
// [rp, 2 rp) of one [M, 2 rp] matrix when the fused gate / up launch reads them, else as two packed [M, rp] matrices.
struct SuLayout {
    int64_t up_offset, pitch;
};
SuLayout su_layout(bool fused_fwd, int rp, int64_t M) {
    if (fused_fwd) return {rp, 2 * (int64_t)rp};
    return {M * rp, rp};
}

int check_call(const xq_weight* gate, const xq_weight* up, const xq_weight* down, const xq_mlp_lora* lora, int64_t M,
               const xq_mlp_saved* saved, const char* who, Dims* d) {
    XQ_REQUIRE(gate && up && down && lora && saved, "%s: NULL descriptor", who);
    int rc;
    if ((rc = xq_validate_weight(gate, who)) || (rc = xq_validate_weight(up, who)) || (rc = xq_validate_weight(down, who))) return rc;
    for (const xq_weight* w : {gate, up, down}) {
        XQ_REQUIRE(w->num_experts == 1, "%s: dense weights only", who);
        XQ_REQUIRE(w->format == XQ_FMT_FP8 || w->layout == XQ_LAYOUT_FLAT, "%s: dense weights are FLAT [out, in]", who);
    }
    const int64_t I = gate->rows, H = gate->cols;
    XQ_REQUIRE(up->rows == I && up->cols == H && down->rows == H && down->cols == I,
               "%s: weight shapes do not make an MLP (gate [%lld, %lld], up [%lld, %lld], down [%lld, %lld])", who, (long long)I,
               (long long)H, (long long)up->rows, (long long)up->cols, (long long)down->rows, (long long)down->cols);
    XQ_REQUIRE(H % 64 == 0 && I % 64 == 0, "%s: hidden size %lld and intermediate size %lld must be multiples of 64", who,
               (long long)H, (long long)I);
    XQ_REQUIRE(M >= 0, "%s: negative row count", who);
    XQ_REQUIRE(lora->r >= 0 && lora->r <= 64, "%s: LoRA rank %d out of range [0, 64]", who, lora->r);
    XQ_REQUIRE(lora->dtype == XQ_DT_F32 || lora->dtype == XQ_DT_BF16, "%s: bad lora dtype", who);
    if (lora->r > 0)
        for (int p = 0; p < 3; ++p) XQ_REQUIRE(lora->A[p] && lora->B[p], "%s: LoRA factor %d is NULL", who, p);
    d->M = M; d->H = H; d->I = I; d->r = lora->r; d->rp = r_pad_of(lora->r);
    if (M > 0) XQ_REQUIRE(saved->gate_up && saved->h && (d->rp == 0 || (saved->su_gate_up && saved->su_down)), "%s: a buffer of xq_mlp_saved is NULL", who);
    XQ_REQUIRE(xq_aligned(saved->gate_up, 16) && xq_aligned(saved->h, 16), "%s: gate_up and h of xq_mlp_saved must be 16-byte aligned", who);
    for (int p = 0; p < 3; ++p) XQ_REQUIRE(xq_aligned(lora->bias[p], 8), "%s: bias vectors must be 8-byte aligned", who);
    return XQ_OK;
}

// one region of split-K partial sums and fp32 sums of the SwiGLU passes (stream order)
// (`needed`: what a call must bring; without it what it is told to bring, room for decoded weights of that format, or of any,
// included)
int64_t gemm_part_bytes(const Dims& d, int fmt, bool needed, bool backward) {
    auto part = [&](int64_t rows, int64_t out, int64_t kc) {
        return needed ? tile_gemm_split_bytes(rows, out, kc) : tile_gemm_partial_bytes(fmt, rows, out, kc);
    };
    const int64_t pa = part(d.M, d.I, d.H), pb = part(d.M, d.H, d.I);
    const int64_t ps = d.rp && silu_bwd_nt_supported(d.I, d.rp) ? silu_nt_partial_bytes(d.M, d.I, d.rp) : 0;
    // the dgrad of block-fp8 gate and up as one sum: the contraction is twice as long
    const bool joint = backward && !needed && (fmt < 0 || fmt == XQ_FMT_FP8) && 2 * d.rp <= 64;
    const int64_t p2 = joint ? tile_gemm_partial_bytes(XQ_FMT_FP8, d.M, d.H, 2 * d.I) : 0;
    return std::max(std::max(pa, pb), std::max(ps, p2));
}

// From a block of 32 rows per compute unit on, the forward lays the A factors out as bf16 panels once and forms s * h . A_d^T in
// the pass that writes h (8192 rows, 12288 columns: 142 us against 120 for the elementwise pass and 41 for the product).
// Below, the product is a launch of its own: blocks of 32 rows would leave compute units idle.
bool many_rows(const Dims& d) { return d.rp > 0 && d.M >= 32ll * num_cus() && silu_bwd_nt_supported(d.I, d.rp); }
int64_t fwd_panel_bytes(const Dims& d) {
    if (!d.rp) return 0;
    if (many_rows(d)) return al256(2 * d.rp * d.H * 2) + al256(d.rp * d.I * 2);
    const int64_t gu = 2 * d.rp <= 64 ? lowrank_panel_bytes(1, d.M, 2 * d.rp, d.H) : lowrank_panel_bytes(2, d.M, d.rp, d.H);
    return std::max(gu, lowrank_panel_bytes(1, d.M, d.rp, d.I));
}

int64_t fwd_workspace(const Dims& d, int fmt, bool needed) { return fwd_panel_bytes(d) + al256(gemm_part_bytes(d, fmt, needed, false)) + 512; }

int64_t bwd_workspace(const Dims& d, int fmt, bool needed) {
    const int64_t rp = d.rp ? d.rp : 16;
    // the six factor gradients share a launch: partial sums of all of them (dA of gate and up of twice the rank, or apart)
    const int64_t tn = 3 * tn_partial_bytes(d.M, d.I, rp) + tn_partial_bytes(d.M, d.H, rp) +
                       std::max(2 * tn_partial_bytes(d.M, d.H, rp), 2 * rp <= 64 ? tn_partial_bytes(d.M, d.H, 2 * rp) : 0);
    return al256(d.M * d.I * 2) + al256(d.M * 2 * d.I * 2) + al256(d.M * d.H * 2) + al256(d.M * rp * 2) +
           al256(d.M * 2 * rp * 2) + 2 * al256(rp * d.I * 2) + al256(std::max(gemm_part_bytes(d, fmt, needed, true), tn)) + 512;
}

}  // namespace
}  // namespace xq

using namespace xq;

extern "C" int xq_set_mlp_gate_up_fused(int enabled) {
    g_mlp_gu = enabled != 0;
    return XQ_OK;
}

extern "C" int xq_get_mlp_gate_up_fused(void) { return g_mlp_gu.load() != 0; }

extern "C" int xq_mlp_gate_up_joint(const xq_weight* gate, const xq_weight* up, int64_t M) {
    if (!gate || !up || M <= 0 || xq_validate_weight(gate, "xq_mlp_gate_up_joint") || xq_validate_weight(up, "xq_mlp_gate_up_joint")) return 0;
    return gate_up_side_by_side(gate, up, nullptr, gate->cols, M, nullptr, nullptr, nullptr, 2 * gate->rows);
}

extern "C" int64_t xq_mlp_workspace_bytes_fmt(int format, int64_t M, int64_t hidden, int64_t intermediate, int r, int backward) {
    if (M < 0 || r < 0) return 0;
    Dims d{M, hidden, intermediate, r, r_pad_of(r)};
    return backward ? bwd_workspace(d, format, false) : fwd_workspace(d, format, false);
}
extern "C" int64_t xq_mlp_workspace_bytes(int64_t M, int64_t hidden, int64_t intermediate, int r, int backward) {
    return xq_mlp_workspace_bytes_fmt(-1, M, hidden, intermediate, r, backward);
}

extern "C" int xq_mlp_fwd(const xq_weight* gate, const xq_weight* up, const xq_weight* down, const xq_mlp_lora* lora,
                          const void* x_, int64_t ldx, int64_t M, void* y, int64_t ldy, xq_mlp_saved* saved,
                          void* workspace, int64_t workspace_bytes, void* stream_) {
    static const char* who = "xq_mlp_fwd";
    Dims d;
    int rc = check_call(gate, up, down, lora, M, saved, who, &d);
    if (rc) return rc;
    const bool fused = fuse_gate_up_fwd(gate, up, saved->gate_up_fused);
    saved->gate_up_fused = fused ? 1 : 0;       // what the backward must be told
    if (M == 0) return XQ_OK;
    XQ_REQUIRE(x_ && y, "%s: NULL activation pointer", who);
    XQ_REQUIRE(workspace && xq_aligned(workspace, 256) && workspace_bytes >= fwd_workspace(d, -1, true),
               "%s: workspace missing, misaligned or smaller than xq_mlp_workspace_bytes()", who);
    XQ_REQUIRE(ldy % 8 == 0 && xq_aligned(y, 16), "%s: y rows must be 16-byte aligned", who);
    // (before anything runs, and for whichever launches read them)
    XQ_REQUIRE(d.rp == 0 || (xq_aligned(saved->su_gate_up, 16) && xq_aligned(saved->su_down, 16)),
               "%s: su_gate_up and su_down of xq_mlp_saved must be 16-byte aligned", who);
    hipStream_t stream = (hipStream_t)stream_;
    const bf16_t* x = (const bf16_t*)x_;
    const int r = d.r, rp = d.rp;
    const int64_t H = d.H, I = d.I;
    const float s = lora->scaling;
    bf16_t *gu = (bf16_t*)saved->gate_up, *h = (bf16_t*)saved->h;
    bf16_t *su_gu = (bf16_t*)saved->su_gate_up, *su_d = (bf16_t*)saved->su_down;
    Carve cv{(uint8_t*)workspace, 0};
    const SuLayout sl = su_layout(fused, rp, M);
    const int f32 = lora->dtype == XQ_DT_F32;
    auto right_of = [&](int p) { return LowRankRight{{lora->B[p], nullptr}, r, r, rp, f32, 0}; };
    const LowRankRight right_g = right_of(0), right_u = right_of(1), right_d = right_of(2);
    FactorMode fm = factor_mode(lora->dtype, false);
    bf16_t* panels = cv.take<bf16_t>(fwd_panel_bytes(d));
    const void *A_g = lora->A[0], *A_u = lora->A[1];
    const bool many = many_rows(d) && !fused;
    float* part = cv.take<float>(0);
    const int64_t part_bytes = workspace_bytes - cv.used;
    bf16_t* A_d = panels + 2 * (int64_t)rp * H;
    int ra = r;                                   // ranks in the factors the products read
    if (many) {
        PanelJobs pj{};
        pj.in_f32 = f32;
        A_g = pj.add(lora->A[0], 1, r, H, false, panels, 1, rp, H);
        A_u = pj.add(lora->A[1], 1, r, H, false, panels + (int64_t)rp * H, 1, rp, H);
        pj.add(lora->A[2], 1, r, I, false, A_d, 1, rp, I);
        if ((rc = launch_panel_prep(pj, stream))) return rc;
        fm = kFacBf16;
        ra = rp;
    }
    if (rp) {
        // bf16(s * x . A^T) of gate and up: one pass over x where both factors fit one
        const LowRankJob both{x, ldx, H, {A_g, A_u}, 2, ra, rp, s, su_gu, sl.pitch, sl.up_offset};
        const LowRankJob apart[2] = {{x, ldx, H, {A_g, nullptr}, 1, ra, rp, s, su_gu, sl.pitch, 0},
                                     {x, ldx, H, {A_u, nullptr}, 1, ra, rp, s, su_gu + sl.up_offset, sl.pitch, 0}};
        rc = 2 * rp <= 64 ? launch_lowrank(&both, 1, M, fm, panels, stream, part, part_bytes) : launch_lowrank(apart, 2, M, fm, panels, stream);
        if (rc) return rc;
    }
    const bf16_t *bias_g = (const bf16_t*)lora->bias[0], *bias_u = (const bf16_t*)lora->bias[1], *bias_d = (const bf16_t*)lora->bias[2];
    if (fused) {
        if ((rc = launch_gate_up_swiglu(gate, up, x, ldx, M, rp ? su_gu : nullptr, rp ? su_gu + sl.up_offset : nullptr, sl.pitch,
                                        LowRankRight{{lora->B[0], lora->B[1]}, r, r, rp, f32, 0}, rp, bias_g, bias_u, gu, 2 * I, h, I, stream)))
            return rc;
    } else {
        if (gate_up_side_by_side(gate, up, x, ldx, M, bias_g, bias_u, gu, 2 * I)) {      // (what it does not take, two launches take or refuse)
            if ((rc = launch_gate_up(gate, up, x, ldx, M, su_gu, rp ? su_gu + sl.up_offset : nullptr, sl.pitch, LowRankRight{{lora->B[0], lora->B[1]}, r, r, rp, f32, 0}, rp,
                                     bias_g, bias_u, gu, 2 * I, stream, who))) return rc;
        } else {
            if ((rc = launch_tile_gemm(gate, true, x, ldx, M, nullptr, nullptr, rp ? su_gu : nullptr, nullptr, rp, bias_g, gu, 2 * I, stream, who, part, part_bytes, nullptr, rp ? &right_g : nullptr, SumOrder::kept))) return rc;
            if ((rc = launch_tile_gemm(up, true, x, ldx, M, nullptr, nullptr, rp ? su_gu + sl.up_offset : nullptr, nullptr, rp, bias_u, gu + I, 2 * I, stream, who, part, part_bytes, nullptr,
                                       rp ? &right_u : nullptr, SumOrder::kept))) return rc;
        }
        if (many) {
            if ((rc = launch_silu_fwd_nt(gu, gu + I, 2 * I, h, I, M, I, A_d, rp, s, su_d, rp, stream))) return rc;
        } else if ((rc = xq_silu_mul_fwd(gu, gu + I, 2 * I, nullptr, h, I, M, I, stream))) {
            return rc;
        }
    }
    if (rp && !many) {
        const LowRankJob jd{h, I, I, {lora->A[2], nullptr}, 1, r, rp, s, su_d, rp, 0};
        if ((rc = launch_lowrank(&jd, 1, M, fm, panels, stream, part, part_bytes))) return rc;
    }
    return launch_tile_gemm(down, true, h, I, M, nullptr, nullptr, rp ? su_d : nullptr, nullptr, rp, bias_d, (bf16_t*)y, ldy, stream,
                            who, part, part_bytes, nullptr, rp ? &right_d : nullptr, SumOrder::kept);
}

// ---- forward only: nothing is kept for a backward, so up to 64 rows each projection is free to take the kernel that suits the
// row count (the weight-streaming kernels, gate and up as one launch); beyond, the program of xq_mlp_fwd is the fastest one
// and runs with the buffers it would keep in the workspace
static int64_t infer_linear_ws(int64_t M, int64_t H, int64_t I, int r) {
    const int64_t b = xq_linear_workspace_bytes(M, H, I, r);
    int64_t a = xq_linear_workspace_bytes(M, I, H, r);
    if (M <= 64) {                                // gate and up side by side in a joint launch
        const int64_t joint = 2 * skinny_workspace_bytes(M, I, H, r_pad_of(r));
        a = a > joint ? a : joint;
    }
    return al256((a > b ? a : b) > 2048 ? (a > b ? a : b) : 2048);
}

static int64_t infer_workspace(int fmt, int64_t M, int64_t hidden, int64_t intermediate, int r, bool needed) {
    if (M < 0 || r < 0) return 0;
    const int64_t act = al256(M * 2 * intermediate * 2) + al256(M * intermediate * 2);
    const int64_t program = al256(M * 2 * r_pad_of(r) * 2) + al256(M * r_pad_of(r) * 2) + fwd_workspace(Dims{M, hidden, intermediate, r, r_pad_of(r)}, fmt, needed);
    const int64_t apart = M <= 64 ? infer_linear_ws(M, hidden, intermediate, r) : 0;
    return act + (program > apart ? program : apart) + 256;
}
extern "C" int64_t xq_mlp_infer_workspace_bytes_fmt(int format, int64_t M, int64_t hidden, int64_t intermediate, int r) {
    return infer_workspace(format, M, hidden, intermediate, r, false);
}
extern "C" int64_t xq_mlp_infer_workspace_bytes(int64_t M, int64_t hidden, int64_t intermediate, int r) {
    return infer_workspace(-1, M, hidden, intermediate, r, false);
}

extern "C" int xq_mlp_fwd_infer(const xq_weight* gate, const xq_weight* up, const xq_weight* down, const xq_mlp_lora* lora,
                                const void* x, int64_t ldx, int64_t M, void* y, int64_t ldy, void* workspace,
                                int64_t workspace_bytes, void* stream) {
    static const char* who = "xq_mlp_fwd_infer";
    XQ_REQUIRE(workspace && xq_aligned(workspace, 256), "%s: workspace missing or misaligned", who);
    Dims d;
    Carve cv{(uint8_t*)workspace, 0};
    // (the argument checks are those of xq_mlp_fwd; the buffers it would keep for a backward live in the workspace here)
    xq_mlp_saved tmp{workspace, workspace, workspace, workspace, 0, 0};
    int rc = check_call(gate, up, down, lora, M, &tmp, who, &d);
    if (rc) return rc;
    if (M == 0) return XQ_OK;
    XQ_REQUIRE(x && y, "%s: NULL activation pointer", who);
    XQ_REQUIRE(workspace_bytes >= infer_workspace(-1, M, d.H, d.I, d.r, true),
               "%s: workspace smaller than xq_mlp_infer_workspace_bytes()", who);
    bf16_t* gu = cv.take<bf16_t>(M * 2 * d.I * 2);
    bf16_t* h = cv.take<bf16_t>(M * d.I * 2);
    if (!(skinny_supported(gate, M) || skinny_supported(up, M) || skinny_supported(down, M))) {
        bf16_t* su_gu = cv.take<bf16_t>(M * 2 * d.rp * 2);
        bf16_t* su_d = cv.take<bf16_t>(M * d.rp * 2);
        xq_mlp_saved own{gu, h, su_gu, su_d, -1, 0};
        void* program_ws = cv.take<uint8_t>(0);
        return xq_mlp_fwd(gate, up, down, lora, x, ldx, M, y, ldy, &own, program_ws, workspace_bytes - cv.used, stream);
    }
    void* ws = cv.take<uint8_t>(0);
    const int64_t ws_bytes = workspace_bytes - cv.used;
    xq_linear_job jobs[2] = {
        {gate, lora->A[0], lora->B[0], d.r, lora->scaling, lora->bias[0], gu, 2 * d.I},
        {up, lora->A[1], lora->B[1], d.r, lora->scaling, lora->bias[1], gu + d.I, 2 * d.I},
    };
    // up to 64 rows outside the one-launch kernel: gate and up in one streaming launch whose epilogue writes h
    const SkinnyRowsJob gu_jobs[2] = {
        {gate, lora->A[0], lora->B[0], d.r, lora->scaling, (const bf16_t*)lora->bias[0], h, d.I},
        {up, lora->A[1], lora->B[1], d.r, lora->scaling, (const bf16_t*)lora->bias[1], h, d.I},
    };
    if (skinny_takes_stream(gate, M, ldx, lora->A[0], lora->B[0], lora->dtype, d.r) && skinny_takes_stream(up, M, ldx, lora->A[1], lora->B[1], lora->dtype, d.r) &&
        ldx % 8 == 0 && xq_aligned(x, 16) && skinny_stream_multi_supported(gu_jobs, 2, M)) {
        if ((rc = launch_skinny_stream(gu_jobs, 2, true, (const bf16_t*)x, ldx, M, lora->dtype, ws, (hipStream_t)stream))) return rc;
        XQ_CHECK_LAUNCH(who);
        return xq_linear_fwd(down, h, d.I, M, lora->A[2], lora->B[2], lora->dtype, d.r, lora->scaling, lora->bias[2], y, ldy, nullptr, ws,
                             ws_bytes, stream);
    }
    if ((rc = xq_linear_fwd_multi(jobs, 2, x, ldx, M, lora->dtype, ws, ws_bytes, stream))) return rc;
    if ((rc = xq_silu_mul_fwd(gu, gu + d.I, 2 * d.I, nullptr, h, d.I, M, d.I, stream))) return rc;
    return xq_linear_fwd(down, h, d.I, M, lora->A[2], lora->B[2], lora->dtype, d.r, lora->scaling, lora->bias[2], y, ldy, nullptr, ws,
                         ws_bytes, stream);
}

extern "C" int xq_mlp_bwd(const xq_weight* gate, const xq_weight* up, const xq_weight* down, const xq_mlp_lora* lora,
                          const void* x_, int64_t ldx, const void* dy_, int64_t lddy, int64_t M, const xq_mlp_saved* saved,
                          void* dx, int64_t lddx, const xq_mlp_grads* grads, void* workspace, int64_t workspace_bytes,
                          void* stream_) {
    static const char* who = "xq_mlp_bwd";
    Dims d;
    int rc = check_call(gate, up, down, lora, M, saved, who, &d);
    if (rc) return rc;
    const int r = d.r, rp = d.rp;
    const int64_t H = d.H, I = d.I;
    XQ_REQUIRE(saved->gate_up_fused == 0 || (saved->gate_up_fused == 1 && gate->format == XQ_FMT_FP8 && up->format == XQ_FMT_FP8),
               "%s: xq_mlp_saved::gate_up_fused is %d: pass the struct the forward filled (0 or 1; 1 only for block-fp8 gate and up)", who,
               saved->gate_up_fused);
    XQ_REQUIRE(rp == 0 || grads, "%s: grads is NULL", who);
    if (rp) for (int p = 0; p < 3; ++p) XQ_REQUIRE(grads->dA[p] && grads->dB[p], "%s: a factor gradient buffer is NULL", who);
    hipStream_t stream = (hipStream_t)stream_;
    if (M == 0) {
        for (int p = 0; p < 3 && rp; ++p) {
            const int64_t in = p == 2 ? I : H, outw = p == 2 ? H : I;
            if ((rc = launch_zero_fill(grads->dA[p], (int64_t)r * in * 4, stream))) return rc;
            if ((rc = launch_zero_fill(grads->dB[p], outw * r * 4, stream))) return rc;
        }
        return XQ_OK;
    }
    XQ_REQUIRE(x_ && dy_, "%s: NULL activation pointer", who);
    XQ_REQUIRE(workspace && xq_aligned(workspace, 256) && workspace_bytes >= bwd_workspace(d, -1, true),
               "%s: workspace missing, misaligned or smaller than xq_mlp_workspace_bytes()", who);
    XQ_REQUIRE(!dx || (lddx % 8 == 0 && xq_aligned(dx, 16)), "%s: dx rows must be 16-byte aligned", who);
    const bf16_t *x = (const bf16_t*)x_, *dy = (const bf16_t*)dy_;
    const float s = lora->scaling;
    const bf16_t *gu = (const bf16_t*)saved->gate_up, *h = (const bf16_t*)saved->h;
    const bf16_t *su_gu = (const bf16_t*)saved->su_gate_up, *su_d = (const bf16_t*)saved->su_down;
    const int rp2 = 2 * rp;
    // one dgrad launch for gate and up (block-fp8, side term of width 2 rp)
    const bool fused = two_dense_supported(gate) && two_dense_supported(up) && rp2 <= 64;

    Carve cv{(uint8_t*)workspace, 0};
    const int f32 = lora->dtype == XQ_DT_F32;
    const FactorMode ft = factor_mode(lora->dtype, true);
    // right-hand factors of the dgrads: A^T of down, and of gate and up (side by side in the launch over both)
    const LowRankRight right_d{{lora->A[2], nullptr}, I, r, rp, f32, 1}, right_gu{{lora->A[0], lora->A[1]}, H, r, rp, f32, 1},
        right_g{{lora->A[0], nullptr}, H, r, rp, f32, 1}, right_u{{lora->A[1], nullptr}, H, r, rp, f32, 1};
    bf16_t* dh = cv.take<bf16_t>(M * I * 2);
    bf16_t* dgu = cv.take<bf16_t>(M * 2 * I * 2);         // [M, 2I]: dgate | dup
    bf16_t* dx_u = cv.take<bf16_t>(M * H * 2);            // unfused dgrads: the up projection's share of dX
    bf16_t* v_d = cv.take<bf16_t>(M * (rp ? rp : 16) * 2);
    bf16_t* v_gu = cv.take<bf16_t>(M * (rp ? rp2 : 32) * 2);
    bf16_t* Bt_g = cv.take<bf16_t>((int64_t)(rp ? rp : 16) * I * 2);    // panels of the gate and up factors (many rows)
    bf16_t* Bt_u = cv.take<bf16_t>((int64_t)(rp ? rp : 16) * I * 2);
    float* part = cv.take<float>(0);
    const int64_t part_bytes = workspace_bytes - cv.used;
    bf16_t *dgate = dgu, *dup = dgu + I;

    // ---- down projection
    if (rp) {
        const LowRankJob jd{dy, lddy, H, {lora->B[2], nullptr}, 1, r, rp, s, v_d, rp, 0};
        if ((rc = launch_lowrank(&jd, 1, M, ft, nullptr, stream, part, part_bytes))) return rc;
    }
    if ((rc = launch_tile_gemm(down, false, dy, lddy, M, nullptr, nullptr, rp ? v_d : nullptr, nullptr, rp, nullptr, dh, I, stream, who, part, part_bytes,
                               nullptr, rp ? &right_d : nullptr, SumOrder::kept)))
        return rc;
    // ---- SwiGLU, and s * dgate . B_g^T, s * dup . B_u^T: one pass over (gate, up, dh) where the rank allows, so that the
    // two products do not read dgate | dup back
    const int64_t ld_v = fused ? rp2 : rp;
    bf16_t* v_g = v_gu;
    bf16_t* v_u = fused ? v_gu + rp : v_gu + M * rp;
    const bool one_pass = rp && g_mlp_silu_nt && silu_bwd_nt_supported(I, rp);
    if (one_pass) {
        // every 32 rows read both factors: from 2048 rows on a launch that lays them out as bf16 panels once is the shorter way
        // (8192 rows, r 32: 288 us from the fp32 factors, 206 + 8 from panels; 1000 rows, r 16: 37 against 30 + 6)
        const void *Fg = lora->B[0], *Fu = lora->B[1];
        FactorMode fmode = ft;
        if (M >= 2048) {
            PanelJobs jobs{};
            jobs.in_f32 = f32;
            Fg = jobs.add(lora->B[0], 1, I, r, true, Bt_g, 1, rp, I);
            Fu = jobs.add(lora->B[1], 1, I, r, true, Bt_u, 1, rp, I);
            if ((rc = launch_panel_prep(jobs, stream))) return rc;
            fmode = kFacBf16;
        }
        if ((rc = launch_silu_bwd_nt(gu, gu + I, 2 * I, dh, I, dgate, dup, 2 * I, M, I, Fg, Fu, fmode, fmode == kFacBf16 ? rp : r, rp, s, v_g, v_u, ld_v, part, stream))) return rc;
    } else if ((rc = xq_silu_mul_bwd(gu, gu + I, 2 * I, dh, I, nullptr, dgate, dup, 2 * I, nullptr, M, I, stream))) {
        return rc;
    }
    // ---- gate / up
    if (rp) {
        if (!one_pass) {
            const LowRankJob jv[2] = {{dgate, 2 * I, I, {lora->B[0], nullptr}, 1, r, rp, s, v_g, ld_v, 0}, {dup, 2 * I, I, {lora->B[1], nullptr}, 1, r, rp, s, v_u, ld_v, 0}};
            if ((rc = launch_lowrank(jv, 2, M, ft, nullptr, stream))) return rc;
        }
        // the six factor gradients, one launch: dB[H, r] = dy^T . su_d, dA[r, I] = (h^T . v_d)^T, dB[I, r] of gate and up, dA[r, H] of both
        const SuLayout sl = su_layout(saved->gate_up_fused == 1, rp, M);
        TnJob jobs[6] = {{dy, lddy, H, su_d, rp, rp, r, false, grads->dB[2]},
                         {h, I, I, v_d, rp, rp, r, true, grads->dA[2]},
                         {dgate, 2 * I, I, su_gu, sl.pitch, rp, r, false, grads->dB[0]},
                         {dup, 2 * I, I, su_gu + sl.up_offset, sl.pitch, rp, r, false, grads->dB[1]}};
        int n = 4;
        if (fused) {       // [v_g | v_u]^T . x: one pass over x
            jobs[n++] = TnJob{x, ldx, H, v_gu, rp2, rp2, r, true, grads->dA[0], nullptr, grads->dA[1], rp};
        } else {
            jobs[n++] = TnJob{x, ldx, H, v_g, rp, rp, r, true, grads->dA[0]};
            jobs[n++] = TnJob{x, ldx, H, v_u, rp, rp, r, true, grads->dA[1]};
        }
        if ((rc = launch_tn_multi(jobs, n, M, part, stream))) return rc;
    }
    if (!dx) return XQ_OK;
    if (fused) {
        const TwoBanks two{up, nullptr, nullptr};
        return launch_tile_gemm(gate, false, dgu, 2 * I, M, nullptr, nullptr, rp ? v_gu : nullptr, nullptr, rp2, nullptr, (bf16_t*)dx, lddx,
                                stream, who, part, part_bytes, &two, rp ? &right_gu : nullptr, SumOrder::kept);
    }
    if ((rc = launch_tile_gemm(gate, false, dgate, 2 * I, M, nullptr, nullptr, rp ? v_g : nullptr, nullptr, rp, nullptr, (bf16_t*)dx, lddx, stream, who, part, part_bytes, nullptr,
                               rp ? &right_g : nullptr, SumOrder::kept))) return rc;
    if ((rc = launch_tile_gemm(up, false, dup, 2 * I, M, nullptr, nullptr, rp ? v_u : nullptr, nullptr, rp, nullptr, dx_u, H, stream, who, part, part_bytes, nullptr,
                               rp ? &right_u : nullptr, SumOrder::kept))) return rc;
    add_rows_kernel<<<dim3((unsigned)xq_cdiv(M * (H / 8), 256)), 256, 0, stream>>>((bf16_t*)dx, lddx, dx_u, H, M, H / 8);
    XQ_CHECK_LAUNCH(who);
    return XQ_OK;
}
