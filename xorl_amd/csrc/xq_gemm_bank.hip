// Launches of gemm_bank_kernel (xq_gemm_bank.h): a file of its own, for the time that its programs take to compile.
#include "xq_gemm_bank.h"
#include <atomic>

namespace xq {

template <int FMT, bool CC, bool DENSE>
static int launch_bank_one(const G256Args& args, dim3 grid, hipStream_t s, const char* who) {
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

int launch_bank(const G256Args& f, int fmt, bool cc, hipStream_t s, const char* who) {
    if (!f.offsets) {
        const dim3 grid((unsigned)(f.tiles_m * f.tiles_n), f.W2 ? 2 : 1);
        return cc ? launch_bank_one<XQ_FMT_FP8, true, true>(f, grid, s, who) : launch_bank_one<XQ_FMT_FP8, false, true>(f, grid, s, who);
    }
    const dim3 grid((unsigned)(f.tiles_m * f.tiles_n));
    if (fmt == XQ_FMT_NVFP4) return cc ? launch_bank_one<XQ_FMT_NVFP4, true, false>(f, grid, s, who) : launch_bank_one<XQ_FMT_NVFP4, false, false>(f, grid, s, who);
    return cc ? launch_bank_one<XQ_FMT_FP8, true, false>(f, grid, s, who) : launch_bank_one<XQ_FMT_FP8, false, false>(f, grid, s, who);
}

}  // namespace xq
