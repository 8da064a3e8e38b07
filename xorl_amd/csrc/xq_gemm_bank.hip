// Launches of gemm_bank_kernel (xq_gemm_bank.h): a file of its own, for the time that its programs take to compile.
#include "xq_gemm_bank.h"
#include <atomic>

namespace xq {

template <int FMT, bool CC, bool DENSE, typename Args>
static int launch_bank_one(const Args& args, dim3 grid, hipStream_t s, const char* who) {
    using D = GeoBank<FMT>;
    static std::atomic<bool> attr_set{false};   // the attribute call is idempotent: a race only repeats it
    if (!attr_set) {
        const hipError_t e = hipFuncSetAttribute((const void*)gemm_bank_kernel<FMT, CC, DENSE>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)D::lds_bytes());
        if (e != hipSuccess) {
            xq_set_error("%s: cannot raise the dynamic LDS limit: %s", who, hipGetErrorString(e));
            return XQ_ERR_LAUNCH;
        }
        attr_set = true;
    }
    gemm_bank_kernel<FMT, CC, DENSE><<<grid, D::NT, D::lds_bytes(), s>>>(args);
    return XQ_OK;
}

static int launch_bank_dense(const BankPair& p, unsigned products, bool cc, hipStream_t s, const char* who) {
    const dim3 grid((unsigned)(p.of[0].tiles_m * p.of[0].tiles_n), products);
    return cc ? launch_bank_one<XQ_FMT_FP8, true, true>(p, grid, s, who) : launch_bank_one<XQ_FMT_FP8, false, true>(p, grid, s, who);
}
int launch_bank_pair(const G256Args (&f)[2], bool cc, hipStream_t s, const char* who) { return launch_bank_dense(BankPair{{f[0], f[1]}}, 2, cc, s, who); }

int launch_bank(const G256Args& f, int fmt, bool cc, hipStream_t s, const char* who) {
    if (!f.offsets) return launch_bank_dense(BankPair{{f, f}}, 1, cc, s, who);
    const dim3 grid((unsigned)(f.tiles_m * f.tiles_n));
    if (fmt == XQ_FMT_NVFP4) return cc ? launch_bank_one<XQ_FMT_NVFP4, true, false>(f, grid, s, who) : launch_bank_one<XQ_FMT_NVFP4, false, false>(f, grid, s, who);
    return cc ? launch_bank_one<XQ_FMT_FP8, true, false>(f, grid, s, who) : launch_bank_one<XQ_FMT_FP8, false, false>(f, grid, s, who);
}

}  // namespace xq
