// Values -> 4-bit codes, for the quantizers and the re-quantising merge.
#pragma once
#include "xq_common.h"

namespace xq {

// e2m1 code of a = v4 / 4, clamped to [-6, 6], in the reference encoder's rule (ops/quantize/fp4_codec.py:12-19): codes up to 3
// from trunc(2a + 0.5) with the sum rounded in fp32, then 4 from a >= 1.75 and one more from 2.5, 3.5 and 5.  All of them are
// integer thresholds of w = fl(4a + 1) = 2 fl(2a + 0.5) -- 2, 4, 6, 8, 11, 15, 21, the sum being exact from a = 1 on --, so the
// code is the number of them at or below trunc(w): a population count.  10 instructions against 15 for the comparisons one
// by one (scaling by 4 is exact: the caller folds it into the scale).  A NaN has code 0 (v_med3 takes the least of the others).
__device__ __forceinline__ uint32_t fp4_code4(float v4) {
    constexpr uint32_t kAt = (1u << 2 | 1u << 4 | 1u << 6 | 1u << 8 | 1u << 11 | 1u << 15 | 1u << 21) >> 1;   // (no threshold at 0)
    const uint32_t u = (uint32_t)(__builtin_amdgcn_fmed3f(fabsf(v4), 0.0f, 24.0f) + 1.0f);
    return (uint32_t)__builtin_popcount(kAt & ((1u << u) - 1u)) + (v4 < 0.0f ? 8u : 0u);
}

// NF4: the number of midpoints between neighbouring levels strictly below v (ops/quantize/nf4_codec.py:42-64), v in [-1, 1].
// 32 buckets of width 1/16 hold at most one midpoint each and none lies within 0.02 of a bucket's width of its edge, so the
// bucket's count of midpoints before it plus one comparison is the code whichever way the bucket index rounds.  The 256-byte
// table in LDS is free of bank conflicts for any mix of buckets.  6 instructions against 30.
struct Nf4Bucket {
    float mid;
    uint32_t before;
};

__device__ __forceinline__ Nf4Bucket nf4_bucket(int b) {
    constexpr float kMid[15] = {(float)-0.8480964004993439, (float)-0.6106329262256622, (float)-0.4599952697753906,
                                (float)-0.3396794348955154, (float)-0.2346074059605598, (float)-0.1379117332398891,
                                (float)-0.0455250181257725, (float)0.0397901497781277,  (float)0.1202552504837513,
                                (float)0.2035212516784668,  (float)0.2920137718319893,  (float)0.3893125355243683,
                                (float)0.5016634166240692,  (float)0.6427869200706482,  (float)0.8614784181118012};
    const float lo = (float)(b - 16) * 0.0625f, hi = lo + 0.0625f;
    Nf4Bucket r = {2.0f, 0u};
#pragma unroll
    for (int i = 0; i < 15; ++i) {
        if (kMid[i] < lo) ++r.before;
        else if (kMid[i] < hi) r.mid = kMid[i];
    }
    return r;
}

__device__ __forceinline__ uint32_t nf4_code(float v, const Nf4Bucket* table) {
    const int b = (int)__builtin_fmaf(v, 16.0f, 16.0f);          // 0 .. 32
    const Nf4Bucket k = table[b < 31 ? b : 31];
    return k.before + (v > k.mid ? 1u : 0u);
}

}  // namespace xq
