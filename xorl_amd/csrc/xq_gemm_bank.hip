// Launch of gemm_bank_kernel (xq_gemm_bank.h): a file of its own, for the time that its program takes to compile.
#include "xq_gemm_bank.h"
#include <atomic>

namespace xq {

template <bool CC>
static int launch_bank_one(const G256Args& f, hipStream_t s, const char* who) {
    static std::atomic<bool> attr_set{false};   // the attribute call is idempotent: a race only repeats it
    if (!attr_set) {
        const hipError_t e = hipFuncSetAttribute((const void*)gemm_bank_kernel<CC>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)GeoBank::lds_bytes());
        if (e != hipSuccess) {
            xq_set_error("%s: cannot raise the dynamic LDS limit: %s", who, hipGetErrorString(e));
            return XQ_ERR_LAUNCH;
        }
        attr_set = true;
    }
    gemm_bank_kernel<CC><<<dim3((unsigned)(f.tiles_m * f.tiles_n)), GeoBank::NT, GeoBank::lds_bytes(), s>>>(f);
    return XQ_OK;
}

int launch_bank(const G256Args& f, bool cc, hipStream_t s, const char* who) {
    return cc ? launch_bank_one<true>(f, s, who) : launch_bank_one<false>(f, s, who);
}

}  // namespace xq
