// Host entry points of the fused dequant-GEMM + LoRA path (dense and grouped).
#include "xq_gemm_tile.h"
#include <algorithm>
#include <atomic>
#include "xq_gemm_256.h"
#include "xq_gemm_bank.h"
#include "xq_gemm_dec.h"
#include "xq_gemm_mid.h"
#include <stdlib.h>
#include <mutex>
#include "xq_lora.h"
#include "xq_skinny.h"

namespace xq {

template <int FMT, int LAYOUT>
static void launch_tile_cc(const TileArgs& g, bool contract_cols, dim3 grid, hipStream_t s) {
    if (contract_cols) gemm_tile_kernel<FMT, LAYOUT, true><<<grid, 256, 0, s>>>(g);
    else gemm_tile_kernel<FMT, LAYOUT, false><<<grid, 256, 0, s>>>(g);
}

// kernel-selection policy (xq_set_tile_policy): 0 = by problem size, 1 = always the generic single-buffered
// tile kernel, 2 / 3 = the pipelined kernel with 256x256 / 128x128 tiles whenever the format allows it.
// XQ_SKINNY=0 disables the M <= 64 path.  Both are process-wide test switches: set them while no other thread is
// inside the library.
static int g_skinny_enabled = [] { const char* e = getenv("XQ_SKINNY"); return e ? atoi(e) : 1; }();
static int g_tile_policy = [] { const char* e = getenv("XQ_TILE_POLICY"); return e ? atoi(e) : 0; }();

template <typename K>
static int raise_lds_limit(K kernel, size_t bytes, const char* who) {
    hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if (e != hipSuccess) {
        xq_set_error("%s: cannot raise the dynamic LDS limit: %s", who, hipGetErrorString(e));
        return XQ_ERR_LAUNCH;
    }
    return XQ_OK;
}

template <int FMT, bool CC, bool GROUPED, int T, bool SPLIT256 = false>
static int launch_256_one(const G256Args& f, dim3 grid, hipStream_t s, const char* who) {
    static std::atomic<bool> attr_set{false};   // per instantiation; the attribute call is idempotent: a race only repeats it
    if (!attr_set) {
        int rc = raise_lds_limit(gemm_256_kernel<FMT, CC, GROUPED, T, SPLIT256>, Geo<T>::lds_bytes(CC), who);
        if (rc) return rc;
        attr_set = true;
    }
    gemm_256_kernel<FMT, CC, GROUPED, T, SPLIT256><<<grid, Geo<T>::NT, Geo<T>::lds_bytes(CC), s>>>(f);
    return XQ_OK;
}

// Block-fp8 launches on large unsplit tiles run gemm_dtl16_kernel (dense) and gemm_bank_kernel (expert banks, some dense ones; 1, the default)
// or gemm_256_kernel (0): a process-wide switch for tests and A/B measurements, XQ_FP8_DIRECT in the environment sets it at load time.
static std::atomic<int> g_fp8_direct{[] { const char* e = getenv("XQ_FP8_DIRECT"); return e ? atoi(e) : 1; }()};

constexpr int64_t kDtlMaxK = 2ll * GeoDtl::SCL_MAX * GeoDtl::BK;      // the longest contraction that gemm_dtl16_kernel takes

static int launch_dtl16(const G256Args& f, bool cc, dim3 grid, hipStream_t s, const char* who) {
    static std::atomic<bool> attr_set{false};
    if (!attr_set) {
        int rc = raise_lds_limit(gemm_dtl16_kernel<true>, GeoDtl::lds_total(), who);
        if (!rc) rc = raise_lds_limit(gemm_dtl16_kernel<false>, GeoDtl::lds_total(), who);
        if (rc) return rc;
        attr_set = true;
    }
    if (cc) gemm_dtl16_kernel<true><<<grid, GeoDtl::NT, GeoDtl::lds_total(), s>>>(f);
    else gemm_dtl16_kernel<false><<<grid, GeoDtl::NT, GeoDtl::lds_total(), s>>>(f);
    return XQ_OK;
}

template <int FMT, bool CC, bool GROUPED>
static int launch_256_t(const G256Args& f, int T, dim3 grid, hipStream_t s, const char* who) {
    if constexpr (!GROUPED)
        if (T == 256 && f.ksplit > 1) return launch_256_one<FMT, CC, false, 256, true>(f, grid, s, who);
    return T == 256 ? launch_256_one<FMT, CC, GROUPED, 256>(f, grid, s, who) : launch_256_one<FMT, CC, GROUPED, 128>(f, grid, s, who);
}

template <int FMT>
static int launch_256(const G256Args& f, bool cc, bool grouped, int T, dim3 grid, hipStream_t s, const char* who) {
    if (cc) return grouped ? launch_256_t<FMT, true, true>(f, T, grid, s, who) : launch_256_t<FMT, true, false>(f, T, grid, s, who);
    return grouped ? launch_256_t<FMT, false, true>(f, T, grid, s, who) : launch_256_t<FMT, false, false>(f, T, grid, s, who);
}

// compute units of the current device (256 on MI355X), asked once
int num_cus() {
    static std::atomic<int> cached{0};
    int c = cached.load(std::memory_order_relaxed);
    if (c > 0) return c;
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
        n = 256;
    cached.store(n, std::memory_order_relaxed);
    return n;
}

// Grid of the persistent program (large unsplit tiles): one block per compute unit, a multiple of 8 so that every
// tile of a block falls into the same XCD's range of the tile order; more blocks when a block would otherwise walk
// more tiles than it keeps a table for.  XQ_PERSIST=0 launches one block per tile (same kernel, same results).
static int g_persist = [] { const char* e = getenv("XQ_PERSIST"); return e ? atoi(e) : 1; }();
static inline unsigned persistent_grid(int64_t tiles) {
    if (!g_persist) return (unsigned)tiles;
    int64_t blocks = std::max<int64_t>((num_cus() / 8) * 8, 8);
    blocks = std::max(blocks, (xq_cdiv(tiles, G256_MAX_ROUNDS) + 7) / 8 * 8);
    return (unsigned)std::min(tiles, blocks);
}

// Tile size of a dense launch under the default policy: large tiles from the point where they fill more than
// half the chip (two small tiles are resident per compute unit, and finish sooner than a half-empty round of
// large ones).
static inline int dense_tile_size(int64_t n_rows, int64_t Nout) {
    return xq_cdiv(n_rows, 256) * xq_cdiv(Nout, 256) > num_cus() / 2 ? 256 : 128;
}

// The same for expert banks.  256 x 256 tiles where an expert's rows fill them (its last tile is half empty on average, and a
// 4-bit tile decodes in full) and the tiles there are fill half the chip.  Forward and backward of a routed MLP, large over small tiles, by rows an
// expert: 4-bit banks, 64 or 128 experts 93 1.15, 187 1.04 to 1.08, 281 1.03 to 1.10, 421 0.97 to 0.99, 656 0.93; 16 experts 250
// 1.10 to 1.14, 500 0.90; 8 experts 500 1.09 to 1.14, 750 0.87.  Block-fp8: 64 or 128 experts 46 1.14, 62 1.01, 93 1.04, 125 0.91, 281 0.87; 16
// experts 125 1.00, 250 0.98, 500 0.81; 8 experts 125 1.23, 250 0.94, 750 0.87.
// `bank_tiles`, products of gemm_bank_kernel whose sums are free: its 128 x 256 tiles, two on a compute unit, where there is one for every compute unit, half a tile an
// expert left empty, or for two in five where an expert's rows fill half of one (nvfp4) or most of one.  Routed MLP forward and backward, all
// their products on these tiles, over 128 x 128 tiles, by rows an expert, block-fp8: 128 experts 2048/768 8 0.96, 24 0.95, 56 0.86, 96 0.84; 64 experts 2048/1024 6
// 0.94, 16 0.95, 32 1.03, 64 0.92, 96 0.81; 64 experts 1280/640 6 1.10 and 16 1.02 (175 and 200 tiles), 32 0.99, 64 0.94; 32 experts 4096/1536 6
// 1.01, 32 1.03, 64 0.88; 32 experts 1536/640 56 1.02, 72 1.02 (150 and 170 tiles), 96 0.97; 16 experts 2560/1024 40 1.11, 72 1.06 (136 tiles),
// 96 0.95; over 256 x 256 tiles, one on a compute unit: 128 experts 128 0.83, 300 0.87, 512 0.91, 1024 0.91; 16 experts 192 0.94, 512 0.90.
// nvfp4, over the tiles of nf4's rule: 128 experts 2048/768 6 0.85, 16 0.87, 32 0.81, 64 0.76, 128 0.73, 256 0.71, 600 0.77; 64 experts 1280/640 16
// 1.05, 32 0.99 (240 tiles), 64 0.91, 128 0.88, 600 0.78; 16 experts 2560/1024 32 1.05, 64 0.98 (128 tiles), 96 0.89, 256 0.82, 600 0.81.
// (Tiles are counted without the empty part of an expert's last column tile: forwards of 8 and 16 experts 2816/1152, whose 1152 columns are
// four and a half, block-fp8 90 tiles 1.12, 108 0.98, 130 0.95; nvfp4 90 1.15, 108 0.97, 130 0.91; 16 experts 1536/640 100 1.04 and 1.13.)
static inline bool bank_large_tiles(int fmt, int64_t n_rows, int num_experts, int64_t Nout, bool bank_tiles) {
    if (bank_tiles) {
        using D = GeoBank<XQ_FMT_FP8>;
        const int64_t tiles = (xq_cdiv(n_rows, D::ROWS) + num_experts / 2) * Nout / D::COLS;
        return tiles >= (n_rows >= (fmt == XQ_FMT_FP8 ? 90ll : 60ll) * num_experts ? num_cus() * 13 / 32 : num_cus());
    }
    const int64_t tiles = (xq_cdiv(n_rows, 256) + num_experts / 2) * xq_cdiv(Nout, 256);
    return n_rows >= (fmt == XQ_FMT_FP8 ? 100ll : 400ll) * num_experts && tiles > num_cus() / 2;
}

// K splits of a dense launch of `blocks` tiles of size T over nk K-steps (1 = none): used when the tiles fill at
// most half of the block slots of the chip (256 large tiles, 512 small ones); every split keeps at least 8 K-steps.
static inline int ksplit_for(int64_t blocks, int T, int64_t nk) {
    const int64_t slots = T == 256 ? num_cus() : 2 * num_cus();   // one large or two small tiles per compute unit
    if (blocks <= 0 || blocks * 2 > slots) return 1;
    int64_t s = slots / blocks;
    if (s > nk / 8) s = nk / 8;
    if (s > 8) s = 8;
    return s < 2 ? 1 : (int)s;
}

// How the default policy runs a dense [n_rows, Nout] product over nk K-steps: `head_rows` leading rows on tiles of
// size T in `split` K splits, and, when head_rows < n_rows, the trailing rows as a second launch.  A launch of large
// tiles whose last round would fill only part of the chip keeps the tile rows that make whole rounds and hands the
// others either to small tiles (two of those blocks share a CU) or to large tiles in K splits, whichever the
// estimates below make cheaper; the whole launch stays as it is unless that saves a fifth of a round.
struct DensePlan {
    int T, split;
    int64_t head_rows;
    int tail_T, tail_split;
};
static DensePlan plan_dense(int64_t n_rows, int64_t Nout, int64_t nk) {
    DensePlan p{dense_tile_size(n_rows, Nout), 1, n_rows, 0, 1};
    if (p.T == 128) {
        p.split = ksplit_for(xq_cdiv(n_rows, 128) * xq_cdiv(Nout, 128), 128, nk);
        return p;
    }
    const int64_t tr = xq_cdiv(n_rows, 256), tc = xq_cdiv(Nout, 256), cus = num_cus();
    const int64_t full = tr * tc / cus, rem = tr * tc - full * cus;
    const int64_t keep = full * cus / tc;                  // tile rows that stay on whole rounds of large tiles
    if (rem == 0 || keep == 0 || keep >= tr) return p;
    const int64_t tail_rows = n_rows - keep * 256;
    // costs in units of one round of large tiles (measured: small tiles take 0.54 of it with up to one block per
    // CU, 0.7 with up to two; a split large tile 1/S of it plus the pass over its fp32 partial sums at ~4 TB/s,
    // a round lasting ~1.9 us per K-step)
    const int64_t n128 = xq_cdiv(tail_rows, 128) * xq_cdiv(Nout, 128);
    const double small_cost = n128 <= cus ? 0.54 : 0.7 * (double)xq_cdiv(n128, 2 * cus);
    const int s256 = ksplit_for((tr - keep) * tc, 256, nk);
    const double round_us = 1.9 * (double)nk;
    const double split_cost = s256 > 1 ? 1.0 / s256 + (3.0 + (4.0 * s256 + 2.0) * (double)tail_rows * (double)Nout / 4.0e6) / round_us : 1e9;
    const double tail_cost = small_cost < split_cost ? small_cost : split_cost;
    if ((double)xq_cdiv(keep * tc, cus) + tail_cost < (double)(full + 1) - 0.2) {
        p.head_rows = keep * 256;
        if (split_cost < small_cost) { p.tail_T = 256; p.tail_split = s256; }
        else { p.tail_T = 128; p.tail_split = 1; }
    }
    return p;
}

// Whether a dense block-fp8 product that would run as planned above takes gemm_bank_kernel's 128 x 256 tiles instead, two on a compute
// unit: where the last round of 256 x 256 tiles would fill up to half of the chip, or leave a launch of 128 x 128 tiles.  Its blocks are
// then at most one more on each unit, which runs alone there and half as long again as beside another; past half they are two and
// a whole round.  150 random products of 400 .. 6000 rows, its time over the plan's: whole launches on 256 x 256 tiles whose last round
// is filled to 0.3 .. 0.5 0.80 to 0.93 ([12288, 4096], 2048 rows 204 -> 172 us); to 0.53 1.00 to 1.09, to 0.6 .. 0.9 1.00 to 1.08.  Two
// launches, the second of 128 x 128 tiles: 0.77 to 0.99, 0.86 in the mean ([7552, 512], 2595 rows 43.9 -> 33.9 us).  Where K splits take the
// last round (0.90 to 1.07), or gemm_mid_kernel the product (0.86 to 1.14), neither is the better.
// Contractions of 192 and 256 likewise (24 products, 0.79 to 0.95), and up to an eighth of a round beyond whole ones (48 products over 192 .. 1536
// k, 0.85 to 0.98).  (A few rows beyond whole tile rows, over such a short contraction, keep the two launches: the form that a test asks for by its
// sizes, [4096, 256], 4100 rows 34.3 us, 32.2 here.)
// The sums are gemm_dtl16_kernel's, whose place these tiles take in a whole launch; rows that would be a launch of 128 x 128 tiles are summed in
// another order (gemm_256_kernel).
static bool half_tiles(const DensePlan& p, int64_t n_rows, int64_t Nout, int64_t Kc, SumOrder order) {
    using D = GeoBank<XQ_FMT_FP8>;
    if (p.T != 256 || p.split != 1 || (Kc <= 256 && p.head_rows < n_rows && n_rows - p.head_rows <= 16)) return false;
    if (order == SumOrder::kept && p.head_rows < n_rows) return false;
    if (p.head_rows < n_rows) return p.tail_T == 128;
    const int64_t blocks = xq_cdiv(n_rows, D::ROWS) * xq_cdiv(Nout, D::COLS), slots = 2ll * num_cus();
    return blocks > slots && blocks % slots != 0 && blocks % slots <= slots / 2;
}

// ---- dense weights decoded once per launch (xq_gemm_dec.h).  The image costs a pass over the weight (50 M weights: 26-33 us)
// and gives back what the tile kernels lose to their decode: a quarter to a third of a 4-bit launch's time, a tenth of a
// block-fp8 one's (whose kernel keeps the bytes in LDS and decodes beside its MFMAs).  Forward, us, image against tile kernel:
//   int4 [12288, 4096]: 512 rows 92 / 101, 700 115 / 128, 1357 153 / 171, 4096 323 / 403, 8192 636 / 820; [4096, 12288]: 512 114 / 94,
//   700 114 / 143, 8192 627 / 786; [4096, 4096]: 512 55 / 45, 1024 69 / 70, 1357 80 / 96; [1024, 4096]: 2048 50 / 45, 4096 72 / 68,
//   8192 101 / 113; block-fp8 [12288, 4096]: 1357 155 / 145, 4096 335 / 327, 8192 626 / 661; [8192, 5120]: 4096 271 / 267, 8192 518 / 545.
// Block-fp8, forward / dgrad, per cent by which the image is faster (negative: slower), nine weights:
//   rows                        3072       4096       5120       6144       7168       8192       16384
//   [12288, 4096]              1 / 0      2 / 0      4 / 3      5 / 5      6 / 1      6 / 3      5 / 4
//   [4096, 12288]              2 / -2     2 / 0      5 / 2      7 / 4      3 / 4      4 / 4      4 / 4
//   [8192, 5120]               2 / -1     2 / 1      3 / -2     4 / 3      6 / 4      6 / 3      7 / 5
//   [4096, 4096]               1 / 0      2 / 1     10 / 1      5 / 5      6 / 5      5 / 5      7 / 6
//   [2048, 2048]             -13 / -16   -5 / -10    4 / 4      2 / 0      3 / 2      2 / 2      6 / 5
//   [1024, 5120]               1 / -9     0 / -6    17 / -1    12 / -1    10 / -7     8 / 3      6 / 6
//   [1024, 4096]              -3 / -9    -4 / -7    10 / -13    6 / -2     4 / 1      3 / 1      5 / 6
//   [4096, 1024]              -8 / -7    -6 / -9   -11 / 8      0 / 2      1 / 2      2 / 1      5 / 5
//   [512, 4096]              -16 / -14  -13 / -10   -7 / -14   -1 / -12   -3 / -3    -2 / -5     4 / 3
// (256 x 256 tiles on both sides.)  So 4-bit from 640 rows on, block-fp8 from 6144 on (both directions gain but for a narrow dgrad whose
// tiles fill a round badly, and below it the wide weights gain less than the narrow ones lose); products too small to fill the
// chip (2e10: the last line up to 8192 rows) stay with the tile kernels.  Below 6144 rows block-fp8 takes the image where its
// choice of tiles fills the rounds better than 256 x 256 do, by the estimates (us, tile kernel -> image: [4224, 7040], 4147 rows
// 262 -> 206; [3200, 3072], 5572 rows 129 -> 97, dgrad 126 -> 96; [6272, 2432], 2855 rows 106 -> 84; [3840, 9216], 5146 rows 384 -> 297; of
// 180 forwards and dgrads of 640 .. 6143 rows 32 took it, 1.08 to 1.32 times as fast, one of them slower, by 4 per cent).
constexpr int64_t kDecMinRows = 640, kDecMinRowsFp8 = 6144;
constexpr double kDecLeadFp8 = 0.92;                 // what the image's estimate has to stay under, of gemm_dtl16_kernel's
constexpr double kDecMinWork = 2.0e10;               // rows x columns x contraction
// Tiles: 256 x 256 where they fill their rounds of the chip; otherwise the rows or columns of a tile are stretched or cut to what
// leaves the last round fullest (288 tiles on 256 units are 240 of 288 rows).  Forward / dgrad, us, with 256 x 256 alone -> with all five:
//   int4 [12288, 4096], 1357 rows: 148 / 164 -> 133 / 164; [8192 -> 5120], 4096 rows 298 -> 261; [4224 -> 7936], 2063 rows 136 / 186 -> 131 /
//   157; [3712 -> 3200], 5416 rows 132 -> 111; [1536 -> 2816], 7253 rows 82 -> 61; [5248, 2176], 3606 rows 99 / 109 -> 79 / 103;
//   nf4 [2304, 6528], 3675 rows 145 / 117 -> 121 / 110; nvfp4 [6272, 1280], 2709 rows 72 / 67 -> 54 / 67.
// The leads below: two estimates of one product err against each other by up to 5 per cent; 224 rows, whose weight tile is read for
// fewer rows, gave back less than the estimate said (six products of 13 were slower at a lead of 0.97, by up to 6 per cent).
struct DecTile {
    int tm, tn;               // 32 tm rows x 64 tn columns
    double lead;              // what part of the time of the tiles before it its estimate has to stay under
};
static const DecTile kDecTiles[] = {{8, 4, 1.0}, {7, 4, 0.88}, {9, 4, 0.92}, {10, 4, 0.92}, {8, 5, 0.92}};
struct DecPart {
    int64_t rows;
    int tile, split;          // index into kDecTiles; K splits
};
struct DecPlan {
    DecPart part[2];          // leading rows, and the others (0: none) as a second launch
    int64_t partial;          // bytes of fp32 sums the splits take
    double us;                // the estimate it was chosen by
};
static DecPlan make_plan_decoded(int64_t n_rows, int64_t Nout, int64_t Kc, int64_t cus) {
    // microseconds, fitted to 32 products on all five tiles in one to four splits (4.7 per cent rms): a K-step takes longer the more of
    // the chip is at work (the matrix units share its power), by the tile's size; the fp32 sums of splits are written and read at
    // about 6 TB/s
    const int64_t steps = Kc / GeoDec::BK;
    auto cost = [&](int tile, int64_t rows, int s) {
        const DecTile t = kDecTiles[tile];
        const double w = (double)(t.tm * t.tn) / 32.0, st = (double)xq_cdiv(steps, s) * w;
        const int64_t blocks = xq_cdiv(rows, 32 * t.tm) * xq_cdiv(Nout, 64 * t.tn) * s, full = blocks / cus, rest = blocks % cus;
        const double sums = s > 1 ? std::max(2.0, 0.165e-6 * (8.0 * s + 2.0) * (double)rows * (double)Nout - 4.6) : 0.0;
        auto round = [&](double f) { return st * (0.423 + 0.288 * f) + 6.2 * w; };
        return (double)full * round(1.0) + (rest ? round((double)rest / (double)cus) : 0.0) + sums;
    };
    auto best = [&](int64_t rows, DecPart* p) {
        *p = DecPart{rows, 0, 1};
        double c = cost(0, rows, 1);
        for (int tile = 0; tile < (int)(sizeof(kDecTiles) / sizeof(kDecTiles[0])); ++tile)
            for (int s = 1; s == 1 || (s <= 8 && steps / s >= 16); ++s) {
                const double lead = tile == p->tile ? 1.0 : kDecTiles[tile].lead, u = cost(tile, rows, s);
                if (u < lead * c) { *p = DecPart{rows, tile, s}; c = u; }
            }
        return c;
    };
    DecPlan p{};
    p.us = best(n_rows, &p.part[0]);
    const int64_t tc = xq_cdiv(Nout, GeoDec::T), tr = xq_cdiv(n_rows, GeoDec::T), keep = tr * tc / cus * cus / tc;      // tile rows of whole rounds
    if (keep > 0 && keep < tr) {
        DecPart tail;
        const double c = cost(0, keep * GeoDec::T, 1) + best(n_rows - keep * GeoDec::T, &tail) + 4.0;
        if (c < p.us) {
            p.part[0] = DecPart{keep * GeoDec::T, 0, 1};
            p.part[1] = tail;
            p.us = c;
        }
    }
    for (const DecPart& d : p.part)
        if (d.split > 1) p.partial = std::max(p.partial, d.split * d.rows * Nout * 4);
    return p;
}
static DecPlan plan_decoded(int64_t n_rows, int64_t Nout, int64_t Kc) {
    static thread_local PlanSlot<DecPlan> kept[64];
    const PlanKey key{n_rows, Nout, Kc, num_cus(), 0};
    PlanSlot<DecPlan>& e = kept[key.slot()];
    if (!(e.key == key)) e = PlanSlot<DecPlan>{key, make_plan_decoded(n_rows, Nout, Kc, key.cus)};
    return e.value;
}
static double decoded_us(int fmt, int64_t n_rows, int64_t Nout, int64_t Kc) {      // with the pass that writes the image
    return 3.4 + (fmt == XQ_FMT_NF4 ? 0.5e-6 : 0.43e-6) * (double)Nout * (double)Kc + plan_decoded(n_rows, Nout, Kc).us;
}
// gemm_dtl16_kernel's 256 x 256 tiles as plan_dense lays them out
static double direct_us(int64_t n_rows, int64_t Nout, int64_t Kc) {
    const int64_t nk = Kc / 64, cus = num_cus();
    const DensePlan p = plan_dense(n_rows, Nout, nk);
    auto us = [&](int64_t rows, int T, int s) {
        if (rows <= 0) return 0.0;
        const int64_t blocks = xq_cdiv(rows, T) * xq_cdiv(Nout, T) * s;
        const double sums = s > 1 ? std::max(2.0, 0.165e-6 * (8.0 * s + 2.0) * (double)rows * (double)Nout - 4.6) : 0.0;
        if (T == 128) return 4.0 + (blocks <= cus ? 0.54 : 0.7 * (double)xq_cdiv(blocks, 2 * cus)) * 1.55 * (double)nk;
        const int64_t full = blocks / cus, rest = blocks % cus;
        const double st = (double)xq_cdiv(nk, s);
        return (double)full * (8.0 + 1.55 * st) + (rest ? 8.0 + (0.9 + 0.65 * (double)rest / (double)cus) * st : 0.0) + sums;
    };
    return us(p.head_rows, 256, p.split) + us(n_rows - p.head_rows, p.tail_T, p.tail_split);
}
static bool decode_first(int fmt, int64_t n_rows, int64_t Nout, int64_t Kc) {
    if (n_rows < kDecMinRows || (double)n_rows * (double)Nout * (double)Kc < kDecMinWork || Kc % 64 != 0 || Kc < 128 || Nout % 16 != 0) return false;
    if (fmt != XQ_FMT_FP8 || n_rows >= kDecMinRowsFp8) return true;
    return dense_tile_size(n_rows, Nout) == 256 && decoded_us(fmt, n_rows, Nout, Kc) < kDecLeadFp8 * direct_us(n_rows, Nout, Kc);
}
// (fmt < 0: whatever the format; the 4-bit rule covers all)
static int64_t decoded_scratch_bytes(int fmt, int64_t n_rows, int64_t Nout, int64_t Kc) {
    return decode_first(fmt < 0 ? XQ_FMT_INT4 : fmt, n_rows, Nout, Kc) ? dec_image_bytes(Nout, Kc) + plan_decoded(n_rows, Nout, Kc).partial : 0;
}

// ---- products that gemm_mid_kernel (xq_gemm_mid.h) takes.  Estimates in microseconds, each within about 5 per cent of what was
// measured (four formats, rows 80 .. 3000, weights [4096, 4096], [12288, 4096], [1024, 4096] and [2560, 8192], both directions); the
// launch goes to the kernel with the shorter one.  70 random products of 65 .. 4096 rows over the formats, both directions: 1.16
// times as fast in the mean, up to 1.8.  There is no upper end to the rows: of 438 random products of 3000 .. 8192
// rows 60 came here (256 .. 2176 columns), at 0.69 to 1.00 of the tile kernels' time, 0.85 in the mean.  Forward / dgrad, this kernel against the tile kernels (from 640 rows on 4-bit:
// over decoded images):
//   [4096, 4096]    rows       100          256          512         1024         2048         3000
//   int4             21.3 / 24.9  26.5 / 31.2  35.0 / 42.6  44.6 / 63.0  63.8 / 84.7  103.9 / 89.6 (forward)
//                    21.7 / 24.2  26.0 / 30.1  34.3 / 39.3  45.8 / 60.4  67.6 / 81.0  106.0 / 90.8 (dgrad)
//   block-fp8        20.1 / 21.2  24.0 / 28.2  33.0 / 37.8  42.5 / 56.2  63.5 / 79.9  101.4 / 90.9 (forward)
//   nf4              27.2 / 26.7  33.5 / 33.3  43.9 / 47.4  64.3 / 72.1  87.2 / 81.8  153.4 / 91.5 (forward)
//   [12288, 4096], 512 rows: int4 forward 56.8 / 93.8, dgrad 64.1 / 82.5; block-fp8 54.8 / 73.9, 61.3 / 71.2
struct MidPlan {
    int mw, split;
    double us;
};
static MidPlan plan_mid(int fmt, bool cc, int64_t rows, int64_t Nout, int64_t Kc) {
    // a step of 64 k and both phases takes c + d f, f the share of the compute units that are at work
    static const double kStep[3][3][2] = {{{0.93, 0.24}, {1.05, 0.34}, {1.20, 0.45}},       // int4, nvfp4: MW = 2, 3, 4
                                          {{0.75, 0.25}, {0.88, 0.36}, {1.05, 0.47}},       // block-fp8
                                          {{1.95, 0.18}, {2.00, 0.36}, {2.20, 0.32}}};      // nf4 (its level look-ups)
    const int ws = cc && fmt != XQ_FMT_FP8 ? 2 : 1, kind = fmt == XQ_FMT_FP8 ? 1 : fmt == XQ_FMT_NF4 ? 2 : 0;
    const int64_t units = Kc / 64 / ws, cus = num_cus();
    MidPlan best{0, 1, 0.0};
    for (int mw = 2; mw <= 4; ++mw)
        for (int s = 1; s <= 8 && (s == 1 || units * ws >= 4 * s); ++s) {
            const int64_t blocks = xq_cdiv(rows, 32 * mw) * xq_cdiv(Nout, 256) * s, rounds = xq_cdiv(blocks, cus);
            const double f = rounds > 1 ? 1.0 : (double)blocks / (double)cus, *c = kStep[kind][mw - 2];
            const double sums = s > 1 ? 2.0 + 0.18e-6 * (8.0 * s + 2.0) * (double)rows * (double)Nout : 0.0;
            const double us = (double)rounds * (5.5 + 1.15 * mw + (double)(xq_cdiv(units, 2 * s) * ws) * (c[0] + c[1] * f)) + sums;
            if (best.mw == 0 || us < best.us) best = MidPlan{mw, s, us};
        }
    return best;
}
// the same product without it: over a decoded image, or on 256- or 128-row tiles
static double tile_kernels_us(int fmt, int64_t rows, int64_t Nout, int64_t Kc) {
    if (decode_first(fmt, rows, Nout, Kc)) return decoded_us(fmt, rows, Nout, Kc);
    const double nk = (double)(Kc / 64);
    if (dense_tile_size(rows, Nout) == 256) {
        const int64_t tiles = xq_cdiv(rows, 256) * xq_cdiv(Nout, 256), cus = num_cus(), full = tiles / cus;
        const double per = fmt == XQ_FMT_FP8 ? 1.0 : 1.25;
        return full ? ((double)full + (tiles % cus ? 0.7 : 0.0)) * (8.0 + per * 1.55 * nk) : 8.0 + per * (0.9 + 0.65 * (double)tiles / (double)cus) * nk;
    }
    static const double k128[3][4] = {{25.3, 0.61, 0.66, 0.15}, {22.9, 0.29, 0.77, 0.136}, {24.5, 0.77, 0.78, 0.142}};
    const double* c = k128[fmt == XQ_FMT_FP8 ? 1 : fmt == XQ_FMT_NF4 ? 2 : 0];
    const int64_t tiles = xq_cdiv(rows, 128) * xq_cdiv(Nout, 128);
    const int s = ksplit_for(tiles, 128, Kc / 64);
    const double st = (double)xq_cdiv(Kc / 64, s);
    return c[0] + st * (c[1] + c[2] * (double)(tiles * s) / (2.0 * num_cus())) + (s > 1 ? -13.0 + c[3] * 1e-6 * (8.0 * s + 2.0) * (double)rows * (double)Nout : 0.0);
}
static bool mid_shape(int fmt, bool cc, int64_t rows, int64_t Nout, int64_t Kc) {
    // whole units of the contraction for both phases; 4-bit dgrads: whole 16-byte pieces of 32 columns, whole scale groups
    const int64_t unit = cc && fmt != XQ_FMT_FP8 ? 128 : 64;
    // (block-fp8 forwards below 384 k are few steps between two ends, and level with the tile kernels'.  Five widths of 512 .. 8192 under 65 .. 5000
    // rows, us, tile kernels -> here: 960 k 1.10 to 1.37 times as fast ([4096, 960], 512 rows 15.1 -> 13.0), 768 k 1.11 to 1.29, 512 k 1.06 to
    // 1.19, 320 k 0.95 to 1.08, 256 k 0.94 to 1.07, 192 k 0.88 to 1.02)
    return rows > 64 && Kc % unit == 0 && Kc >= (cc && fmt == XQ_FMT_FP8 ? 384 : 2 * unit) &&
           (fmt != XQ_FMT_FP8 || Kc <= 64 * 2 * GeoMid<XQ_FMT_FP8, true, 4>::SCL_MAX) &&
           (cc || fmt == XQ_FMT_FP8 || Nout % (fmt == XQ_FMT_INT4 ? 128 : 64) == 0) && Nout >= 64;
}
static bool takes_mid(int fmt, bool cc, int64_t rows, int64_t Nout, int64_t Kc, MidPlan* plan) {
    if (!mid_shape(fmt, cc, rows, Nout, Kc)) return false;
    struct Answer { MidPlan plan; bool taken; };
    static thread_local PlanSlot<Answer> kept[64];
    const PlanKey key{rows, Nout, Kc, num_cus(), fmt * 2 + (cc ? 1 : 0)};
    PlanSlot<Answer>& e = kept[key.slot()];
    if (e.key == key) {
        *plan = e.value.plan;
        return e.value.taken;
    }
    *plan = plan_mid(fmt, cc, rows, Nout, Kc);
    // (a lead the estimates can carry: over random shapes a smaller one was a loss as often as a gain, up to 8 per cent for nf4)
    const double lead = fmt == XQ_FMT_NF4 ? 0.94 : !decode_first(fmt, rows, Nout, Kc) && dense_tile_size(rows, Nout) == 256 ? 0.94 : 0.98;
    e = PlanSlot<Answer>{key, Answer{*plan, plan->us < lead * tile_kernels_us(fmt, rows, Nout, Kc)}};
    return e.value.taken;
}
static int64_t mid_partial_bytes(int fmt, bool cc, int64_t rows, int64_t Nout, int64_t Kc) {
    MidPlan p;
    return takes_mid(fmt, cc, rows, Nout, Kc, &p) && p.split > 1 ? p.split * rows * Nout * 4 : 0;
}

extern "C" int xq_dense_route(int format, int forward, int64_t rows, int64_t n_out, int64_t k, int32_t plan[6]) {
    if (format < XQ_FMT_INT4 || format > XQ_FMT_NF4 || rows <= 0 || n_out <= 0 || k <= 0 || k % BK || n_out % 16) return -1;
    for (int i = 0; i < 6; ++i) plan[i] = 0;
    auto put = [&](int part, int tile_rows, int tile_cols, int split) {
        plan[3 * part] = tile_rows;
        plan[3 * part + 1] = tile_cols;
        plan[3 * part + 2] = split;
    };
    MidPlan mid;
    if (takes_mid(format, forward != 0, rows, n_out, k, &mid)) {
        put(0, 32 * mid.mw, 256, mid.split);
        return XQ_ROUTE_MID;
    }
    if (decode_first(format, rows, n_out, k)) {
        const DecPlan p = plan_decoded(rows, n_out, k);
        for (int i = 0; i < 2; ++i)
            if (p.part[i].rows > 0) put(i, 32 * kDecTiles[p.part[i].tile].tm, 64 * kDecTiles[p.part[i].tile].tn, p.part[i].split);
        return XQ_ROUTE_IMAGE;
    }
    const DensePlan p = plan_dense(rows, n_out, k / BK);
    if (format == XQ_FMT_FP8 && half_tiles(p, rows, n_out, k, SumOrder::any)) {
        put(0, GeoBank<XQ_FMT_FP8>::ROWS, GeoBank<XQ_FMT_FP8>::COLS, 1);
        return XQ_ROUTE_TILES;
    }
    put(0, p.T, p.T, p.split);
    if (p.head_rows < rows) put(1, p.tail_T, p.tail_T, p.tail_split);
    return XQ_ROUTE_TILES;
}

// fp32 partial-sum bytes the split-K forms of a dense [n_rows, Nout] product over Kc may want, under any tile policy
int64_t tile_gemm_split_bytes(int64_t n_rows, int64_t Nout, int64_t Kc) {
    if (n_rows <= 0 || Kc % BK) return 0;
    const int64_t nk = Kc / BK;
    int64_t elems = 0;
    for (int T : {128, 256}) {         // a whole launch on either tile size (default or forced policy)
        const int s = ksplit_for(xq_cdiv(n_rows, T) * xq_cdiv(Nout, T), T, nk);
        if (s > 1 && s * n_rows > elems) elems = s * n_rows;
    }
    const DensePlan p = plan_dense(n_rows, Nout, nk);
    if (p.head_rows < n_rows && p.tail_split > 1 && p.tail_split * (n_rows - p.head_rows) > elems)
        elems = p.tail_split * (n_rows - p.head_rows);
    return elems * Nout * 4;
}

// scratch a dense launch of this format (< 0: of any) may want: the above, or the decoded image of the weight with the sums of
// its splits (without room for those the launch decodes in the tile kernel)
int64_t tile_gemm_partial_bytes(int fmt, int64_t n_rows, int64_t Nout, int64_t Kc) {
    if (n_rows <= 0 || Kc % BK) return 0;
    int64_t mid = 0;
    for (int f : {XQ_FMT_INT4, XQ_FMT_NVFP4, XQ_FMT_FP8, XQ_FMT_NF4})
        if (fmt < 0 || fmt == f)
            for (bool cc : {true, false}) mid = std::max(mid, mid_partial_bytes(f, cc, n_rows, Nout, Kc));
    return std::max(mid, std::max(tile_gemm_split_bytes(n_rows, Nout, Kc), decoded_scratch_bytes(fmt, n_rows, Nout, Kc)));
}

// Whether a grouped launch on this bank may take a second bank of the same shape (see G256Args::W2): block-fp8 on the
// pipelined kernel, whole 256-column tiles per bank (which also keeps the K-step where the dgrad changes banks on a
// scale-block boundary and away from the pipeline's prologue).
bool two_banks_supported(const xq_weight* w) {
    return w->format == XQ_FMT_FP8 && g_tile_policy != 1 && w->cols % 256 == 0 && w->cols >= 512 && w->num_experts >= 1;
}

// Whether gemm_bank_kernel takes a product over kc of rows of A within span_rows, lda apart: dense block-fp8, block-fp8 banks and nvfp4 banks in their
// usual storage, three K-steps, an output in whole 16-byte pieces, operands within 32-bit byte offsets of a base (up to 3 KB further on).
// Kept sums are gemm_dtl16_kernel's, block-fp8 as far as that kernel goes.  (nvfp4 banks under a forced tile size stay on gemm_256_kernel, whose
// sums are the same for both sizes.)
static bool bank_kernel_takes(const xq_weight* w, bool bank, int64_t kc, SumOrder order, int64_t span_rows, int64_t lda, const void* C, int64_t ldc, const void* bias) {
    constexpr int64_t reach = (1ll << 32) - 4096;
    const bool fp8 = w->format == XQ_FMT_FP8 && g_fp8_direct && g_tile_policy != 1 && (order == SumOrder::any || kc <= kDtlMaxK);
    const bool f4 = bank && w->format == XQ_FMT_NVFP4 && w->layout == XQ_LAYOUT_GKN && w->group == 16 && w->scale_dtype == XQ_SCALE_E4M3 &&
                    g_tile_policy == 0 && order == SumOrder::any;
    return (fp8 || f4) && kc % BK == 0 && kc >= 3 * BK && w->cols % 16 == 0 && xq_aligned(w->packed, 16) && w->rows * w->cols < reach && span_rows > 0 &&
           span_rows * lda * 2 < reach && xq_aligned(C, 16) && ldc % 8 == 0 && xq_aligned(bias, 8) && !(bank && bias);
}
// ... as far as the weight says: a bank's product with rows 16-byte aligned and few enough
static bool bank_kernel_takes(const xq_weight* w, int64_t kc, SumOrder order) { return bank_kernel_takes(w, true, kc, order, 1, kc, nullptr, 8, nullptr); }

// tile size of a grouped launch on the pipelined kernel, or (256, where it takes the launch) gemm_bank_kernel
static inline int bank_tile_size(int fmt, int64_t n_rows, int num_experts, int64_t Nout, bool bank_tiles) {
    return g_tile_policy == 2 ? 256 : g_tile_policy == 3 ? 128 : bank_large_tiles(fmt, n_rows, num_experts, Nout, bank_tiles) ? 256 : 128;
}

// ... of two banks' columns side by side: small tiles too where large ones do not divide a bank's columns and one bank alone would not take them
static inline int side_by_side_tile(int fmt, int64_t n_rows, int num_experts, int64_t ncols, bool bank_tiles) {
    const int T = bank_tile_size(fmt, n_rows, num_experts, 2 * ncols, bank_tiles);
    return ncols % T != 0 ? bank_tile_size(fmt, n_rows, num_experts, ncols, bank_tiles) : T;
}

// Whether two 4-bit banks of one shape and storage take one launch whose output holds both products side by side, ncols columns
// each (G256Args::W2): whole column tiles per bank.  One bank's tiles leave half of the block slots empty at some hundreds of
// routed rows and end in a round of their own beyond (routed MLP, two launches and one, us: nf4 32 experts 2560/1024, 800 rows, forward and backward 510 and 461; nvfp4 64 experts 2048/1024, 9000 rows 886 and 816, forward alone of 6000 rows 350 and 305).
bool banks_side_by_side(const xq_weight* a, const xq_weight* b, bool contract_cols, int64_t n_rows, SumOrder order) {
    const int64_t ncols = contract_cols ? a->rows : a->cols;
    const bool free = order == SumOrder::any && bank_kernel_takes(a, contract_cols ? a->cols : a->rows, order);
    return a->format != XQ_FMT_FP8 && tile_gemm_takes_row_map(a) && tile_gemm_takes_row_map(b) && a->format == b->format &&
           a->rows == b->rows && a->cols == b->cols && a->num_experts == b->num_experts && a->group == b->group &&
           a->scale_dtype == b->scale_dtype && xq_packed_bytes_per_expert(a) % 16 == 0 && xq_aligned(a->packed, 16) && xq_aligned(b->packed, 16) &&
           ncols % side_by_side_tile(a->format, n_rows, a->num_experts, ncols, free) == 0;
}

extern "C" int xq_bank_route(const xq_weight* w, int forward, int joint, int kept, int64_t n_rows) {
    if (!w || n_rows <= 0 || xq_validate_weight(w, "xq_bank_route") || !tile_gemm_takes_row_map(w)) return -1;
    const bool one_sum = joint && !forward && w->format == XQ_FMT_FP8;
    const int64_t nout = forward ? w->cols : w->rows, kc = (forward ? w->rows : w->cols) * (one_sum ? 2 : 1);
    const SumOrder order = kept ? SumOrder::kept : SumOrder::any;
    const bool ok = bank_kernel_takes(w, kc, order), free = ok && !kept;
    const int T = joint && w->format != XQ_FMT_FP8 ? side_by_side_tile(w->format, n_rows, w->num_experts, nout, free)
                                                   : bank_tile_size(w->format, n_rows, w->num_experts, nout * (joint && !one_sum ? 2 : 1), free);
    return T == 128 ? XQ_BANK_TILES_128 : ok ? XQ_BANK_HALF_TILES : XQ_BANK_TILES_256;
}

// Whether the dgrad of two dense [N, K] weights of one shape may run as one launch (see launch_tile_gemm): block-fp8 on
// the pipelined kernel, the change of matrix on a scale-block boundary and past the pipeline's prologue.
bool two_dense_supported(const xq_weight* w) {
    return w->format == XQ_FMT_FP8 && g_tile_policy != 1 && w->num_experts == 1 && w->rows % 128 == 0 && w->rows >= 512;
}

template <int TM, int TN>
static int launch_dec_tile(G256Args& f, hipStream_t s, const char* who) {
    using G = GeoDecTile<TM, TN>;
    static std::atomic<bool> attr_set{false};
    if (!attr_set) {
        int rc = raise_lds_limit(gemm_dec_kernel<false, TM, TN>, G::lds_bytes(), who);
        if (!rc) rc = raise_lds_limit(gemm_dec_kernel<true, TM, TN>, G::lds_bytes(), who);
        if (rc) return rc;
        attr_set = true;
    }
    f.tiles_m = (int32_t)xq_cdiv(f.M, G::ROWS);
    f.tiles_n = (int32_t)xq_cdiv(f.Nout, G::COLS);
    const dim3 grid((unsigned)(f.tiles_m * f.tiles_n), (unsigned)f.ksplit);
    if (f.ksplit > 1) gemm_dec_kernel<true, TM, TN><<<grid, GeoDec::NT, G::lds_bytes(), s>>>(f);
    else gemm_dec_kernel<false, TM, TN><<<grid, GeoDec::NT, G::lds_bytes(), s>>>(f);
    XQ_CHECK_LAUNCH(who);
    return XQ_OK;
}

// The launches of a dense weight decoded once: `f` is filled for the whole problem (f.W2: a second matrix that continues the
// contraction), weights FLAT; `scratch` holds decoded_scratch_bytes().
static int launch_decoded(G256Args f, bool cc, int fmt, uint8_t* scratch, hipStream_t stream, const char* who) {
    const DecPlan plan = plan_decoded(f.M, f.Nout, f.Kc);
    bf16_t* image = (bf16_t*)scratch;
    f.partial = (float*)(scratch + dec_image_bytes(f.Nout, f.Kc));
    const int mats = f.W2 ? 2 : 1;
    DecImageArgs im{f.W, f.scales, f.global_scale, f.wrows, f.wcols, f.gshift, f.scale_dtype, f.Kc / mats, f.Nout, image, f.Kc / GeoDec::BK, 0};
    const unsigned tiles_n = (unsigned)xq_cdiv(f.Nout, GeoDec::T);
    const bool timed = xq_profile_mark_begin(stream, 2.0 * (double)f.M * f.Nout * ((double)f.Kc + f.r_pad));
    auto decode = [&](auto FMT_) {
        constexpr int FMT = decltype(FMT_)::value;
        if (cc) dec_image_kernel<FMT><<<dim3((unsigned)xq_cdiv(im.Kc, 256), tiles_n * 8), 256, 0, stream>>>(im);
        else dec_image_t_kernel<FMT><<<dim3((unsigned)(im.Kc / 64), tiles_n), 256, 0, stream>>>(im);
    };
    for (int m = 0; m < mats; ++m) {
        if (m) { im.packed = f.W2; im.scales = f.scales2; im.kt0 = im.Kc / GeoDec::BK; }
        if (fmt == XQ_FMT_FP8) decode(std::integral_constant<int, XQ_FMT_FP8>{});
        else if (fmt == XQ_FMT_INT4) decode(std::integral_constant<int, XQ_FMT_INT4>{});
        else if (fmt == XQ_FMT_NF4) decode(std::integral_constant<int, XQ_FMT_NF4>{});
        else decode(std::integral_constant<int, XQ_FMT_NVFP4>{});
        XQ_CHECK_LAUNCH(who);
    }
    f.W = (const uint8_t*)image;
    const bf16_t *A = f.A, *su = f.su;
    bf16_t* C = f.C;
    int64_t r0 = 0;
    for (const DecPart& part : plan.part) {
        if (part.rows == 0) continue;
        f.M = part.rows;
        f.A = A + r0 * f.lda;
        f.su = su ? su + r0 * f.ld_su : nullptr;
        f.C = C + r0 * f.ldc;
        f.ksplit = part.split;
        r0 += part.rows;
        int rc;
        switch (part.tile) {
            case 0: rc = launch_dec_tile<8, 4>(f, stream, who); break;
            case 1: rc = launch_dec_tile<7, 4>(f, stream, who); break;
            case 2: rc = launch_dec_tile<9, 4>(f, stream, who); break;
            case 3: rc = launch_dec_tile<10, 4>(f, stream, who); break;
            default: rc = launch_dec_tile<8, 5>(f, stream, who);
        }
        if (rc) return rc;
        if (f.ksplit > 1) {
            splitk_reduce_kernel<<<(unsigned)xq_cdiv(f.M * (f.Nout >> 2), 256), 256, 0, stream>>>(f.partial, f.ksplit, f.M, f.Nout, f.C, f.ldc);
            XQ_CHECK_LAUNCH(who);
        }
    }
    if (timed) xq_profile_mark_end(stream);
    return XQ_OK;
}

template <int FMT, bool CC>
static int launch_mid_t(const G256Args& f, int mw, dim3 grid, hipStream_t s, const char* who) {
    static std::atomic<bool> attr_set{false};
    if (!attr_set) {
        int rc = raise_lds_limit(gemm_mid_kernel<FMT, CC, 4>, GeoMid<FMT, CC, 4>::lds_bytes(), who);
        if (!rc) rc = raise_lds_limit(gemm_mid_kernel<FMT, CC, 3>, GeoMid<FMT, CC, 3>::lds_bytes(), who);
        if (!rc) rc = raise_lds_limit(gemm_mid_kernel<FMT, CC, 2>, GeoMid<FMT, CC, 2>::lds_bytes(), who);
        if (rc) return rc;
        attr_set = true;
    }
    if (mw == 4) gemm_mid_kernel<FMT, CC, 4><<<grid, 512, GeoMid<FMT, CC, 4>::lds_bytes(), s>>>(f);
    else if (mw == 3) gemm_mid_kernel<FMT, CC, 3><<<grid, 512, GeoMid<FMT, CC, 3>::lds_bytes(), s>>>(f);
    else gemm_mid_kernel<FMT, CC, 2><<<grid, 512, GeoMid<FMT, CC, 2>::lds_bytes(), s>>>(f);
    return XQ_OK;
}
static int launch_mid(G256Args f, bool cc, int fmt, int mw, hipStream_t s, const char* who) {
    f.tiles_m = (int32_t)xq_cdiv(f.M, 32 * mw);
    f.tiles_n = (int32_t)xq_cdiv(f.Nout, 256);
    const dim3 grid((unsigned)(f.tiles_m * f.tiles_n), (unsigned)f.ksplit);
    const bool timed = xq_profile_mark_begin(s, 2.0 * (double)f.M * f.Nout * ((double)f.Kc + f.r_pad));
    int rc;
    if (fmt == XQ_FMT_FP8) rc = cc ? launch_mid_t<XQ_FMT_FP8, true>(f, mw, grid, s, who) : launch_mid_t<XQ_FMT_FP8, false>(f, mw, grid, s, who);
    else if (fmt == XQ_FMT_INT4) rc = cc ? launch_mid_t<XQ_FMT_INT4, true>(f, mw, grid, s, who) : launch_mid_t<XQ_FMT_INT4, false>(f, mw, grid, s, who);
    else if (fmt == XQ_FMT_NF4) rc = cc ? launch_mid_t<XQ_FMT_NF4, true>(f, mw, grid, s, who) : launch_mid_t<XQ_FMT_NF4, false>(f, mw, grid, s, who);
    else rc = cc ? launch_mid_t<XQ_FMT_NVFP4, true>(f, mw, grid, s, who) : launch_mid_t<XQ_FMT_NVFP4, false>(f, mw, grid, s, who);
    if (rc) return rc;
    XQ_CHECK_LAUNCH(who);
    if (f.ksplit > 1) {
        splitk_reduce_kernel<<<(unsigned)xq_cdiv(f.M * (f.Nout >> 2), 256), 256, 0, s>>>(f.partial, f.ksplit, f.M, f.Nout, f.C, f.ldc);
        XQ_CHECK_LAUNCH(who);
    }
    if (timed) xq_profile_mark_end(s);
    return XQ_OK;
}

// C[rows, Nout] = A . op(deq(W)) (+ su . Lr^T) (+ bias); see xq_gemm_tile.h.  force_T = 256 / 128 fixes the tile
// size of the pipelined kernel (and force_split its K splits), 0 leaves both to the selection policy.  `partial` (may be NULL) is scratch for
// split-K sums; a launch that would split but finds less than tile_gemm_partial_bytes() there runs unsplit.
static int launch_tile_gemm_t(const xq_weight* w, bool contract_cols, const bf16_t* A, int64_t lda, int64_t n_rows,
                              const int32_t* offsets, const int32_t* tile_offsets, const bf16_t* su, const bf16_t* lora_right,
                              int r_pad, const bf16_t* bias, bf16_t* C, int64_t ldc, hipStream_t stream, const char* who,
                              int force_T, int force_split, float* partial, int64_t partial_bytes,
                              const TwoBanks* two = nullptr, const LowRankRight* right = nullptr,
                              SumOrder order = SumOrder::any, const int32_t* a_rows = nullptr, int64_t a_span_rows = 0) {
    const int64_t a_rows_span = a_rows ? a_span_rows : n_rows;      // rows of A that the launch may touch (0: not known)
    TileArgs g;
    g.A = A; g.lda = lda; g.C = C; g.ldc = ldc;
    g.packed = (const uint8_t*)w->packed;
    g.scales = (const uint8_t*)w->scales;
    g.global_scale = w->global_scale;
    g.packed_stride = xq_packed_bytes_per_expert(w);
    g.scale_stride = xq_scale_bytes_per_expert(w);
    g.wrows = (int32_t)w->rows; g.wcols = (int32_t)w->cols;
    g.group = w->group; g.scale_dtype = w->scale_dtype;
    g.Kc = contract_cols ? g.wcols : g.wrows;
    g.Nout = contract_cols ? g.wrows : g.wcols;
    const bool two_dense = two && !offsets;
    if (two) {
        // a second matrix of the same shape.  Expert banks: twice the contraction (dgrad) or twice the output columns
        // (forward).  Dense [N, K] weights: the dgrad contracts over the rows of both, dX = [dY1 | dY2] . [W1 ; W2].
        XQ_REQUIRE(two->w2 && two->w2->rows == w->rows && two->w2->cols == w->cols && two->w2->num_experts == w->num_experts,
                   "%s: a two-matrix launch takes two weights of one shape", who);
        if (two_dense) {
            XQ_REQUIRE(!contract_cols && two_dense_supported(w) && two_dense_supported(two->w2),
                       "%s: the dense two-matrix form is the dgrad of two block-fp8 weights (out_features %% 128 == 0, >= 512)", who);
            g.Kc *= 2;
        } else {
            XQ_REQUIRE((two_banks_supported(w) && two_banks_supported(two->w2)) || banks_side_by_side(w, two->w2, contract_cols, n_rows, order),
                       "%s: a two-bank launch takes two block-fp8 expert banks (columns a multiple of 256) or two 4-bit ones (whole tiles)", who);
            XQ_REQUIRE(xq_aligned(two->su2, 16) && xq_aligned(two->lora_right2, 16) && two->a_off2 % 8 == 0, "%s: the second bank's operands must be 16-byte aligned", who);
            if (contract_cols && w->format == XQ_FMT_FP8) g.Kc *= 2;
            else g.Nout *= 2;
        }
    }
    g.n_rows = n_rows; g.offsets = offsets; g.tile_offsets = tile_offsets; g.num_experts = w->num_experts;
    XQ_REQUIRE(!offsets || !right, "%s: expert banks take their right-hand factors as panels", who);
    XQ_REQUIRE(offsets || !lora_right, "%s: internal error: a dense launch takes the right-hand factor as it is", who);
    g.su = su; g.lora_right = lora_right; g.right = right ? *right : LowRankRight{}; g.r_pad = (su && (lora_right || right)) ? r_pad : 0;
    g.bias = bias;
    XQ_REQUIRE(g.Kc % BK == 0, "%s: contraction length %d must be a multiple of %d", who, g.Kc, BK);
    XQ_REQUIRE(g.Nout % 16 == 0, "%s: output width %d must be a multiple of 16", who, g.Nout);
    XQ_REQUIRE(lda % 8 == 0 && xq_aligned(A, 16), "%s: activation rows must be 16-byte aligned", who);
    XQ_REQUIRE(xq_aligned(w->packed, 16) && g.packed_stride % 16 == 0, "%s: packed weight must be 16-byte aligned", who);
    XQ_REQUIRE(g.r_pad == 0 || (g.r_pad % 16 == 0 && g.r_pad <= 64 && xq_aligned(su, 16) && xq_aligned(lora_right, 16) &&
                                (!right || (right->r >= 1 && right->r <= right->rp && right->rp * (right->f[1] ? 2 : 1) == r_pad))),
               "%s: bad low-rank side term (r_pad %d)", who, g.r_pad);
    if (w->format != XQ_FMT_FP8 && w->layout == XQ_LAYOUT_GKN)
        XQ_REQUIRE(w->rows % 2 == 0, "%s: GKN 4-bit storage needs an even row count", who);
    if (n_rows == 0) return XQ_OK;
    // block-fp8 and FLAT 4-bit weights: the pipelined tile kernel, 256x256 tiles when they fill the chip,
    // 128x128 tiles otherwise (dense or grouped)
    {
        const bool grouped = offsets != nullptr;
        int gshift = 0;
        while ((1 << gshift) < g.group) ++gshift;
        // 4-bit: power-of-two groups of at least 16; dense matrices FLAT, expert banks GKN (16-byte pieces of codes
        // and of scales: columns in multiples of 16, 16-byte aligned scale storage)
        const bool fmt_ok = w->format == XQ_FMT_FP8 ||
                            ((1 << gshift) == g.group && g.group >= 16 &&
                             (grouped ? w->layout == XQ_LAYOUT_GKN && g.wcols % 16 == 0 && g.wrows >= 2 &&
                                            xq_aligned(w->scales, 16) && g.scale_stride % 16 == 0
                                      : w->layout == XQ_LAYOUT_FLAT));
        const DensePlan plan = plan_dense(n_rows, g.Nout, g.Kc / BK);
        const bool planned = !grouped && fmt_ok && g_tile_policy == 0 && force_T == 0 && !two_dense;   // two matrices: one unsplit launch
        const bool bank_ok = fmt_ok && bank_kernel_takes(w, grouped, g.Kc, order, a_rows_span, lda, C, ldc, bias), free = bank_ok && order == SumOrder::any;
        int T = force_T ? force_T : g_tile_policy == 2 ? 256 : g_tile_policy == 3 ? 128 : plan.T;
        if (grouped && two && w->format != XQ_FMT_FP8) {
            T = side_by_side_tile(w->format, n_rows, w->num_experts, g.Nout / 2, free);
            if (g.Nout / 2 % T != 0) T = 128;      // (joined by what the weights say, and rows that span too much for gemm_bank_kernel)
        } else if (grouped) {
            T = bank_tile_size(w->format, n_rows, w->num_experts, g.Nout, free);
        }
        MidPlan mid;
        const bool by_size = planned || (two_dense && g_tile_policy == 0);
        // (its storages: the formats' usual groups and scale types; 32-bit offsets from a base for the operands)
        const bool mid_storage = w->format == XQ_FMT_FP8 || (w->format == XQ_FMT_INT4 && g.group == 128 && g.scale_dtype == XQ_SCALE_BF16) ||
                                 (w->format == XQ_FMT_NVFP4 && g.group == 16 && g.scale_dtype == XQ_SCALE_E4M3) ||
                                 (w->format == XQ_FMT_NF4 && g.group == 64 && g.scale_dtype == XQ_SCALE_F32);
        if (by_size && fmt_ok && mid_storage && (w->format != XQ_FMT_FP8 || g_fp8_direct) && g.wcols % (w->format == XQ_FMT_FP8 ? 16 : g.group) == 0 &&
            takes_mid(w->format, contract_cols, n_rows, g.Nout, g.Kc, &mid) && n_rows * lda * 2 < (1ll << 32) &&
            (int64_t)g.wrows * g.wcols < (1ll << 32) &&
            (mid.split == 1 || (partial && xq_aligned(partial, 16) && partial_bytes >= mid.split * n_rows * g.Nout * 4))) {
            G256Args f{};
            f.A = A; f.lda = lda; f.C = C; f.ldc = ldc;
            f.W = g.packed; f.scales = g.scales; f.global_scale = g.global_scale;
            f.wrows = g.wrows; f.wcols = g.wcols; f.gshift = gshift; f.scale_dtype = g.scale_dtype;
            f.Kc = g.Kc; f.Nout = g.Nout; f.M = n_rows; f.num_experts = 1;
            if (two) { f.W2 = (const uint8_t*)two->w2->packed; f.scales2 = (const uint8_t*)two->w2->scales; f.nk1 = g.wrows / BK; }
            f.su = g.r_pad ? su : nullptr; f.right = g.right; f.r_pad = g.r_pad; f.ld_su = g.r_pad;
            f.bias = bias;
            f.ksplit = mid.split; f.partial = mid.split > 1 ? partial : nullptr;
            f.wide_rows = xq_aligned(C, 16) && ldc % 8 == 0;
            return launch_mid(f, contract_cols, w->format, mid.mw, stream, who);
        }
        if (by_size && (w->format != XQ_FMT_FP8 || g_fp8_direct) &&
            decode_first(w->format, n_rows, g.Nout, g.Kc) && partial && xq_aligned(partial, 16) &&
            partial_bytes >= decoded_scratch_bytes(w->format, n_rows, g.Nout, g.Kc) && n_rows * lda * 2 < (1ll << 32) && xq_cdiv(n_rows, 256) * xq_cdiv(g.Nout, 256) < (1ll << 31) && g.Nout < 65536 * 16) {
            G256Args f{};
            f.A = A; f.lda = lda; f.C = C; f.ldc = ldc;
            f.W = g.packed; f.scales = g.scales; f.global_scale = g.global_scale;
            f.wrows = g.wrows; f.wcols = g.wcols; f.gshift = gshift; f.scale_dtype = g.scale_dtype;
            f.Kc = g.Kc; f.Nout = g.Nout; f.M = n_rows; f.num_experts = 1;
            if (two) { f.W2 = (const uint8_t*)two->w2->packed; f.scales2 = (const uint8_t*)two->w2->scales; }
            f.su = g.r_pad ? su : nullptr; f.right = g.right; f.r_pad = g.r_pad; f.ld_su = g.r_pad;
            f.bias = bias;
            f.wide_rows = xq_aligned(C, 16) && ldc % 8 == 0 && xq_aligned(bias, 8);
            return launch_decoded(f, contract_cols, w->format, (uint8_t*)partial, stream, who);
        }
        if (planned && bank_ok && g.right.f[1] == nullptr && half_tiles(plan, n_rows, g.Nout, g.Kc, order)) {
            using D = GeoBank<XQ_FMT_FP8>;
            G256Args f{};
            f.A = A; f.lda = lda; f.C = C; f.ldc = ldc;
            f.W = g.packed; f.scales = g.scales;
            f.wrows = g.wrows; f.wcols = g.wcols; f.scale_dtype = g.scale_dtype;
            f.Kc = g.Kc; f.Nout = g.Nout; f.M = n_rows; f.num_experts = 1;
            f.su = g.r_pad ? su : nullptr; f.right = g.right; f.r_pad = g.r_pad; f.ld_su = g.r_pad;
            f.bias = bias;
            f.tiles_m = (int32_t)xq_cdiv(n_rows, D::ROWS); f.tiles_n = (int32_t)xq_cdiv(g.Nout, D::COLS);
            f.ksplit = 1; f.wide_rows = 1;
            const bool timed = xq_profile_mark_begin(stream, 2.0 * (double)n_rows * g.Nout * ((double)g.Kc + g.r_pad));
            const int rc = launch_bank(f, w->format, contract_cols, stream, who);
            if (rc) return rc;
            XQ_CHECK_LAUNCH(who);
            if (timed) xq_profile_mark_end(stream);
            return XQ_OK;
        }
        if (planned && plan.head_rows < n_rows) {
            const int64_t head = plan.head_rows;
            const int rc = launch_tile_gemm_t(w, contract_cols, A, lda, head, nullptr, nullptr, su, lora_right, r_pad,
                                              bias, C, ldc, stream, who, 256, 1, nullptr, 0, nullptr, right);
            if (rc) return rc;
            return launch_tile_gemm_t(w, contract_cols, A + head * lda, lda, n_rows - head, nullptr, nullptr,
                                      su ? su + head * r_pad : nullptr, lora_right, r_pad, bias, C + head * ldc, ldc,
                                      stream, who, plan.tail_T, plan.tail_split, partial, partial_bytes, nullptr, right);
        }
        const int64_t tiles_m = xq_cdiv(n_rows, T) + (grouped ? w->num_experts : 0);
        const int64_t tiles_n = xq_cdiv(g.Nout, T);
        if (fmt_ok && g_tile_policy != 1 && tiles_m * tiles_n < (1ll << 31)) {
            G256Args f;
            f.A = A; f.lda = lda; f.a_rows = a_rows; f.C = C; f.ldc = ldc;
            f.W = g.packed; f.scales = g.scales; f.global_scale = g.global_scale;
            f.packed_stride = g.packed_stride; f.scale_stride = g.scale_stride;
            f.wrows = g.wrows; f.wcols = g.wcols; f.gshift = gshift; f.scale_dtype = g.scale_dtype;
            f.Kc = g.Kc; f.Nout = g.Nout; f.M = n_rows;
            f.offsets = offsets;
            f.tile_prefix = !grouped ? nullptr : (T == 256 ? tile_offsets + (w->num_experts + 1) : tile_offsets);
            f.num_experts = w->num_experts;
            f.su = g.r_pad ? su : nullptr; f.lora_right = g.r_pad ? lora_right : nullptr; f.right = g.right; f.r_pad = g.r_pad;
            f.bias = bias;
            f.tiles_m = (int32_t)tiles_m; f.tiles_n = (int32_t)tiles_n;
            int ksplit = grouped || two_dense ? 1 : force_T ? force_split : planned ? plan.split : ksplit_for(tiles_m * tiles_n, T, g.Kc / BK);
            if (ksplit > 1 && (!partial || !xq_aligned(partial, 16) || partial_bytes < (int64_t)ksplit * n_rows * g.Nout * 4)) ksplit = 1;
            f.ksplit = ksplit; f.partial = ksplit > 1 ? partial : nullptr;
            f.W2 = nullptr; f.scales2 = nullptr; f.su2 = nullptr; f.lora_right2 = nullptr; f.ncols1 = 0; f.nk1 = 0; f.a_off2 = 0; f.global_scale2 = nullptr;
            f.ld_su = g.r_pad; f.H = nullptr; f.ldh = 0; f.bias2 = nullptr;
            f.wide_rows = xq_aligned(C, 16) && ldc % 8 == 0 && xq_aligned(bias, 8);
            if (two) {
                f.W2 = (const uint8_t*)two->w2->packed; f.scales2 = (const uint8_t*)two->w2->scales;
                f.su2 = g.r_pad ? two->su2 : nullptr; f.lora_right2 = g.r_pad ? two->lora_right2 : nullptr;
                f.ncols1 = contract_cols ? g.wrows : g.wcols; f.a_off2 = two->a_off2; f.global_scale2 = two->w2->global_scale;
                f.nk1 = (two_dense ? g.wrows : g.wcols) / BK;
            }
            // (the kernel's own rule: large unsplit tiles, except the 4-bit expert banks)
            const bool persistent = T == 256 && ksplit == 1 && !(grouped && w->format != XQ_FMT_FP8);
            dim3 grid(persistent ? persistent_grid(tiles_m * tiles_n) : (unsigned)(tiles_m * tiles_n), (unsigned)ksplit);
            const bool timed = xq_profile_mark_begin(stream, 2.0 * (double)n_rows * g.Nout * ((double)g.Kc + g.r_pad));
            int rc;
            // block-fp8, and nvfp4 banks, on large unsplit tiles: the kernels that bring both operand tiles straight into LDS and decode after the fragment
            // read, one block per tile (dense xq_gemm_dtl.h, expert banks xq_gemm_bank.h)
            // (two matrices: the second one starts on a scale-block boundary of the contraction, or -- two banks side by side -- on a
            // tile boundary of the columns)
            const bool side_by_side = grouped && (!contract_cols || w->format != XQ_FMT_FP8);
            const bool large = T == 256 && ksplit == 1 && (!two || (side_by_side ? f.ncols1 % 256 == 0 : (f.nk1 % 2 == 0 && f.nk1 >= 2)));
            if (large && grouped && bank_ok) {
                using D = GeoBank<XQ_FMT_FP8>;
                f.tiles_m = (int32_t)(xq_cdiv(n_rows, D::ROWS) + w->num_experts);
                f.tiles_n = (int32_t)xq_cdiv(g.Nout, D::COLS);
                f.tile_prefix = tile_offsets;                // (its tiles have 128 rows)
                rc = launch_bank(f, w->format, contract_cols, stream, who);
            } else if (large && !grouped && w->format == XQ_FMT_FP8 && g_fp8_direct && g.Kc >= 3 * BK && g.Kc <= kDtlMaxK &&
                       n_rows * lda * 2 < (1ll << 32) && (int64_t)g.wrows * g.wcols < (1ll << 32))      // (32-bit byte offsets from a base)
                rc = launch_dtl16(f, contract_cols, dim3((unsigned)(tiles_m * tiles_n)), stream, who);
            else if (w->format == XQ_FMT_FP8) rc = launch_256<XQ_FMT_FP8>(f, contract_cols, grouped, T, grid, stream, who);
            else if (w->format == XQ_FMT_INT4) rc = launch_256<XQ_FMT_INT4>(f, contract_cols, grouped, T, grid, stream, who);
            else if (w->format == XQ_FMT_NF4) rc = launch_256<XQ_FMT_NF4>(f, contract_cols, grouped, T, grid, stream, who);
            else rc = launch_256<XQ_FMT_NVFP4>(f, contract_cols, grouped, T, grid, stream, who);
            if (rc) return rc;
            XQ_CHECK_LAUNCH(who);
            if (ksplit > 1) {
                const int64_t quads = n_rows * (g.Nout >> 2);
                splitk_reduce_kernel<<<(unsigned)xq_cdiv(quads, 256), 256, 0, stream>>>(partial, ksplit, n_rows, g.Nout, C, ldc);
                XQ_CHECK_LAUNCH(who);
            }
            if (timed) xq_profile_mark_end(stream);
            return XQ_OK;
        }
    }
    XQ_REQUIRE(!a_rows, "%s: internal error: a row map needs the pipelined tile kernel (see tile_gemm_takes_row_map)", who);
    unsigned mt = (unsigned)(xq_cdiv(n_rows, BM) + (offsets ? w->num_experts : 0));
    dim3 grid(mt, (unsigned)xq_cdiv(g.Nout, BN));
    const bool timed = xq_profile_mark_begin(stream, 2.0 * (double)n_rows * g.Nout * ((double)g.Kc + g.r_pad));
    if (w->format == XQ_FMT_FP8) launch_tile_cc<XQ_FMT_FP8, XQ_LAYOUT_FLAT>(g, contract_cols, grid, stream);
    else if (w->format == XQ_FMT_INT4 && w->layout == XQ_LAYOUT_FLAT) launch_tile_cc<XQ_FMT_INT4, XQ_LAYOUT_FLAT>(g, contract_cols, grid, stream);
    else if (w->format == XQ_FMT_INT4) launch_tile_cc<XQ_FMT_INT4, XQ_LAYOUT_GKN>(g, contract_cols, grid, stream);
    else if (w->format == XQ_FMT_NF4 && w->layout == XQ_LAYOUT_FLAT) launch_tile_cc<XQ_FMT_NF4, XQ_LAYOUT_FLAT>(g, contract_cols, grid, stream);
    else if (w->format == XQ_FMT_NF4) launch_tile_cc<XQ_FMT_NF4, XQ_LAYOUT_GKN>(g, contract_cols, grid, stream);
    else if (w->layout == XQ_LAYOUT_FLAT) launch_tile_cc<XQ_FMT_NVFP4, XQ_LAYOUT_FLAT>(g, contract_cols, grid, stream);
    else launch_tile_cc<XQ_FMT_NVFP4, XQ_LAYOUT_GKN>(g, contract_cols, grid, stream);
    if (timed) xq_profile_mark_end(stream);
    XQ_CHECK_LAUNCH(who);
    return XQ_OK;
}

// gate | up | SwiGLU of a dense block-fp8 MLP in one launch: gu[M, 2I] = (x . deq(Wg)^T + side term | x . deq(Wu)^T +
// side term) and h[M, I] = bf16(silu(gate)) * up from the rounded projections.  Both weights [I, K] block-fp8.
int launch_gate_up_swiglu(const xq_weight* wg, const xq_weight* wu, const bf16_t* x, int64_t ldx, int64_t M,
                          const bf16_t* su_g, const bf16_t* su_u, int64_t ld_su, const LowRankRight& right, int r_pad, const bf16_t* bias_g,
                          const bf16_t* bias_u, bf16_t* gu, int64_t ldgu, bf16_t* h, int64_t ldh, hipStream_t stream) {
    static const char* who = "gate_up_swiglu";
    XQ_REQUIRE(wg->format == XQ_FMT_FP8 && wu->format == XQ_FMT_FP8 && wg->rows == wu->rows && wg->cols == wu->cols,
               "%s: two block-fp8 weights of one shape", who);
    const int64_t I = wg->rows, K = wg->cols;
    XQ_REQUIRE(K % BK == 0 && I % 16 == 0, "%s: in_features %% 64 == 0 and out_features %% 16 == 0", who);
    XQ_REQUIRE(ldx % 8 == 0 && xq_aligned(x, 16) && xq_aligned(wg->packed, 16) && xq_aligned(wu->packed, 16),
               "%s: operands must be 16-byte aligned", who);
    XQ_REQUIRE(ldgu % 8 == 0 && ldh % 8 == 0 && xq_aligned(gu, 16) && xq_aligned(h, 16), "%s: output rows must be 16-byte aligned", who);
    XQ_REQUIRE(xq_aligned(bias_g, 8) && xq_aligned(bias_u, 8), "%s: bias vectors must be 8-byte aligned", who);
    const bool side = su_g && su_u && right.f[0] && right.f[1] && r_pad > 0;
    XQ_REQUIRE(!side || (r_pad % 16 == 0 && r_pad <= 64 && ld_su >= r_pad && ld_su % 8 == 0 && xq_aligned(su_g, 16) &&
                         xq_aligned(su_u, 16)),
               "%s: bad low-rank side term", who);
    if (M == 0) return XQ_OK;
    G256Args f{};
    f.A = x; f.lda = ldx; f.C = gu; f.ldc = ldgu;
    f.W = (const uint8_t*)wg->packed; f.scales = (const uint8_t*)wg->scales;
    f.W2 = (const uint8_t*)wu->packed; f.scales2 = (const uint8_t*)wu->scales;
    f.wrows = (int32_t)I; f.wcols = (int32_t)K; f.scale_dtype = XQ_SCALE_F32;
    f.Kc = (int32_t)K; f.Nout = (int32_t)I; f.M = M;
    f.num_experts = 1;
    f.su = side ? su_g : nullptr; f.su2 = side ? su_u : nullptr; f.ld_su = ld_su;
    f.right = right; f.r_pad = side ? r_pad : 0;
    f.bias = bias_g; f.bias2 = bias_u;
    f.tiles_m = (int32_t)xq_cdiv(M, 256); f.tiles_n = (int32_t)xq_cdiv(I, 128);
    f.ksplit = 1;
    f.H = h; f.ldh = ldh;
    f.wide_rows = 1;
    static std::atomic<bool> attr_set{false};
    if (!attr_set) {
        int rc = raise_lds_limit(gemm_256_kernel<XQ_FMT_FP8, true, false, 256, false, true>, Geo<256>::lds_bytes(true), who);
        if (rc) return rc;
        attr_set = true;
    }
    // flops of the two projections and their side terms
    const bool timed = xq_profile_mark_begin(stream, 2.0 * (double)M * (2.0 * I) * ((double)K + f.r_pad));
    gemm_256_kernel<XQ_FMT_FP8, true, false, 256, false, true>
        <<<dim3(persistent_grid((int64_t)f.tiles_m * f.tiles_n)), Geo<256>::NT, Geo<256>::lds_bytes(true), stream>>>(f);
    XQ_CHECK_LAUNCH(who);
    if (timed) xq_profile_mark_end(stream);
    return XQ_OK;
}

// Whether gate and up of a block-fp8 MLP run as one launch of gemm_bank_kernel: products that gemm_dtl16_kernel would run whole, whose sums are the
// same there.  (Fewer rows, in gemm_mid_kernel or K splits, would gain as well -- 4096/12288, us of the three products, 256 rows 131 -> 108, 768
// rows 284 -> 249 -- but 2e-4 to 4e-4 of y and of every gradient with them.)  The blocks of both, two on a compute unit, share the last round.
// Rounds, and the time of a forward's three products over that of three launches, of random MLPs: 1 .. 1.5 0.88 to 0.93, 1.53 1.04, 1.7 .. 1.9
// 0.99 to 1.00, from two rounds on 0.88 to 0.99.
bool gate_up_side_by_side(const xq_weight* wg, const xq_weight* wu, const bf16_t* x, int64_t ldx, int64_t M, const bf16_t* bias_g,
                          const bf16_t* bias_u, const bf16_t* gu, int64_t ldgu) {
    using D = GeoBank<XQ_FMT_FP8>;
    const int64_t I = wg->rows, K = wg->cols;
    if (g_tile_policy != 0 || wg->format != XQ_FMT_FP8 || wu->format != XQ_FMT_FP8 || wu->rows != I || wu->cols != K || I % 16 != 0 || M <= 64 ||
        ldx % 8 != 0 || !xq_aligned(x, 16) || !bank_kernel_takes(wg, false, K, SumOrder::kept, M, ldx, gu, ldgu, bias_g) ||
        !bank_kernel_takes(wu, false, K, SumOrder::kept, M, ldx, gu, ldgu, bias_u))
        return false;
    MidPlan mid;
    if (takes_mid(XQ_FMT_FP8, true, M, I, K, &mid) || decode_first(XQ_FMT_FP8, M, I, K)) return false;
    const DensePlan p = plan_dense(M, I, K / BK);
    if (p.T != 256 || p.split != 1 || p.head_rows < M) return false;
    const int64_t blocks = 2 * xq_cdiv(M, D::ROWS) * xq_cdiv(I, D::COLS), slots = 2ll * num_cus();
    const double rounds = (double)blocks / (double)slots, part = rounds - (double)(blocks / slots);
    return rounds >= 2.0 || !(part > 0.5 && part < 0.63);
}

// gu[M, 2I] = (x . deq(Wg)^T + side term | x . deq(Wu)^T + side term), gate_up_side_by_side() being true
int launch_gate_up(const xq_weight* wg, const xq_weight* wu, const bf16_t* x, int64_t ldx, int64_t M, const bf16_t* su_g, const bf16_t* su_u,
                   int64_t ld_su, const LowRankRight& right, int r_pad, const bf16_t* bias_g, const bf16_t* bias_u, bf16_t* gu, int64_t ldgu,
                   hipStream_t stream, const char* who) {
    using D = GeoBank<XQ_FMT_FP8>;
    const bool side = r_pad > 0;
    G256Args f{};
    f.A = x; f.lda = ldx; f.C = gu; f.ldc = ldgu; f.ncols1 = (int32_t)wg->rows;
    f.W = (const uint8_t*)wg->packed; f.scales = (const uint8_t*)wg->scales;
    f.W2 = (const uint8_t*)wu->packed; f.scales2 = (const uint8_t*)wu->scales;
    f.wrows = (int32_t)wg->rows; f.wcols = (int32_t)wg->cols; f.scale_dtype = wg->scale_dtype;
    f.Kc = f.wcols; f.Nout = f.wrows; f.M = M; f.num_experts = 1;
    f.su = side ? su_g : nullptr; f.su2 = side ? su_u : nullptr; f.right = right; f.r_pad = r_pad; f.ld_su = ld_su;
    f.bias = bias_g; f.bias2 = bias_u;
    f.tiles_m = (int32_t)xq_cdiv(M, D::ROWS); f.tiles_n = (int32_t)xq_cdiv(f.Nout, D::COLS);
    f.ksplit = 1; f.wide_rows = 1;
    const bool timed = xq_profile_mark_begin(stream, 2.0 * (double)M * (2.0 * wg->rows) * ((double)wg->cols + r_pad));
    const int rc = launch_bank(f, XQ_FMT_FP8, true, stream, who);
    if (rc) return rc;
    XQ_CHECK_LAUNCH(who);
    if (timed) xq_profile_mark_end(stream);
    return XQ_OK;
}

int launch_tile_gemm(const xq_weight* w, bool contract_cols, const bf16_t* A, int64_t lda, int64_t n_rows,
                     const int32_t* offsets, const int32_t* tile_offsets, const bf16_t* su, const bf16_t* lora_right,
                     int r_pad, const bf16_t* bias, bf16_t* C, int64_t ldc, hipStream_t stream, const char* who,
                     float* partial, int64_t partial_bytes, const TwoBanks* two, const LowRankRight* right, SumOrder order,
                     const int32_t* a_rows, int64_t a_span_rows) {
    XQ_REQUIRE(!a_rows || offsets, "%s: a row map goes with a grouped launch", who);
    return launch_tile_gemm_t(w, contract_cols, A, lda, n_rows, offsets, tile_offsets, su, lora_right, r_pad, bias, C, ldc,
                              stream, who, 0, 1, partial, partial_bytes, two, right, order, a_rows, a_span_rows);
}

// whether a grouped launch over this bank runs on the pipelined tile kernel, which can read its activation rows through
// a row map (the conditions of launch_tile_gemm_t)
bool tile_gemm_takes_row_map(const xq_weight* w) {
    if (g_tile_policy == 1) return false;
    if (w->format == XQ_FMT_FP8) return true;
    int gshift = 0;
    while ((1 << gshift) < w->group) ++gshift;
    return (1 << gshift) == w->group && w->group >= 16 && w->layout == XQ_LAYOUT_GKN && w->cols % 16 == 0 && w->rows >= 2 &&
           xq_aligned(w->scales, 16) && xq_scale_bytes_per_expert(w) % 16 == 0;
}

static inline int64_t align256(int64_t b) { return (b + 255) & ~(int64_t)255; }
static inline int r_pad_of(int r) { return r <= 0 ? 0 : ((r + 15) / 16) * 16; }

struct Carver {
    uint8_t* base;
    int64_t used, cap;
    void* take(int64_t bytes) {
        void* p = base ? base + used : nullptr;
        used += align256(bytes);
        return p;
    }
};

}  // namespace xq

using namespace xq;

extern "C" int xq_set_tile_policy(int policy) {
    XQ_REQUIRE(policy >= 0 && policy <= 3, "xq_set_tile_policy: policy %d not in {0, 1, 2, 3}", policy);
    g_tile_policy = policy;
    return XQ_OK;
}

extern "C" int xq_set_skinny_one_launch(int enabled) {
    set_skinny_rows(enabled ? 1 : 0);
    return XQ_OK;
}

extern "C" int xq_set_skinny_gemv(int enabled) {
    set_skinny_gemv(enabled);
    return XQ_OK;
}

extern "C" int xq_set_skinny_spin_limit(int limit) {
    set_skinny_rows_spin_limit(limit);
    return XQ_OK;
}

extern "C" int xq_skinny_reset(void) { return reset_skinny_rows_slots(); }

extern "C" int xq_skinny_status(int* gave_up, int* failed_slots, void* stream) {
    int a = 0, b = 0;
    const int rc = skinny_rows_status(&a, &b, (hipStream_t)stream);
    if (gave_up) *gave_up = a;
    if (failed_slots) *failed_slots = b;
    return rc;
}

extern "C" int xq_set_fp8_direct_tiles(int enabled) {
    g_fp8_direct = enabled != 0;
    return XQ_OK;
}

extern "C" int xq_set_persistent_tiles(int enabled) {
    g_persist = enabled != 0;
    return XQ_OK;
}

// what a call must bring (`needed`) and what it is told to bring (with room for the decoded image of a weight of that format, or
// of any, under many rows)
static int64_t linear_workspace(int fmt, int64_t M, int64_t N, int64_t K, int r, bool needed) {
    auto part = [&](int64_t rows, int64_t out, int64_t kc) {
        return needed ? tile_gemm_split_bytes(rows, out, kc) : tile_gemm_partial_bytes(fmt, rows, out, kc);
    };
    int rp = r_pad_of(r);
    int64_t skinny = M <= 64 ? skinny_workspace_bytes(M, N, K, rp) : 0;
    // scratch of the forward (output N, contraction K) and of the dgrad (output K, contraction N)
    const int64_t pf = align256(part(M, N, K));
    const int64_t pb = align256(part(M, K, N));
    int64_t need = (pf > pb ? pf : pb) + 256;
    if (rp) {
        const int64_t panel = lowrank_panel_bytes(1, M, rp, K);
        int64_t fwd = align256(M * rp * 2) + panel + pf;
        int64_t tn = tn_partial_bytes(M, N, rp) + tn_partial_bytes(M, K, rp);     // the weight-gradient partials reuse the dgrad's region
        int64_t bwd = 2 * align256(M * rp * 2) + panel + (tn > pb ? tn : pb);
        need = (fwd > bwd ? fwd : bwd) + 256;
    }
    return need > skinny ? need : skinny;
}
static int64_t linear_workspace_needed(int64_t M, int64_t N, int64_t K, int r) { return linear_workspace(-1, M, N, K, r, true); }
extern "C" int64_t xq_linear_workspace_bytes(int64_t M, int64_t N, int64_t K, int r) { return linear_workspace(-1, M, N, K, r, false); }
extern "C" int64_t xq_linear_workspace_bytes_fmt(int format, int64_t M, int64_t N, int64_t K, int r) { return linear_workspace(format, M, N, K, r, false); }

static int check_dense(const xq_weight* w, const char* who) {
    int rc = xq_validate_weight(w, who);
    if (rc) return rc;
    XQ_REQUIRE(w->num_experts == 1, "%s: dense entry point takes a single matrix", who);
    XQ_REQUIRE(w->format == XQ_FMT_FP8 || w->layout == XQ_LAYOUT_FLAT, "%s: dense weights are FLAT [N, K]", who);
    return XQ_OK;
}

// whether a forward that keeps nothing for a backward runs on the kernels of few rows, and on which of them
static bool takes_skinny(const xq_weight* w, int64_t M, int64_t ldx, const void* lora_A, const void* lora_B, int lora_dtype, int r) {
    return g_skinny_enabled && skinny_supported(w, M) &&
           (stream_takes_pitch(M, ldx) || (skinny_rows_enabled() && skinny_rows_supported(w, M, lora_A, lora_B, lora_dtype, r)));
}
extern "C" int xq_skinny_route(const xq_weight* w, int64_t M, int64_t ldx, const void* lora_A, const void* lora_B, int lora_dtype, int r, int32_t plan[2]) {
    if (!w || !plan || M < 1 || r < 0 || r > 64 || check_dense(w, "xq_skinny_route")) return -1;
    plan[0] = plan[1] = 0;
    if (!takes_skinny(w, M, ldx, lora_A, lora_B, lora_dtype, r)) return XQ_SKINNY_NONE;
    if (!skinny_takes_stream(w, M, ldx, lora_A, lora_B, lora_dtype, r)) return XQ_SKINNY_ONE_LAUNCH;
    skinny_stream_plan(w, M, plan);
    return XQ_SKINNY_STREAM;
}

extern "C" int xq_linear_fwd(const xq_weight* w, const void* x, int64_t ldx, int64_t M, const void* lora_A,
                             const void* lora_B, int lora_dtype, int r, float scaling, const void* bias_bf16, void* y,
                             int64_t ldy, void* su_out, void* workspace, int64_t workspace_bytes, void* stream_) {
    int rc = check_dense(w, "xq_linear_fwd");
    if (rc) return rc;
    const int64_t N = w->rows, K = w->cols;
    XQ_REQUIRE(M >= 0 && (M == 0 || (x && y)), "xq_linear_fwd: NULL activation pointer");   // an empty batch has no storage
    XQ_REQUIRE(r >= 0 && r <= 64, "xq_linear_fwd: LoRA rank %d out of range [0, 64]", r);
    XQ_REQUIRE(r == 0 || (lora_A && lora_B), "xq_linear_fwd: LoRA factors are NULL");
    XQ_REQUIRE(lora_dtype == XQ_DT_F32 || lora_dtype == XQ_DT_BF16, "xq_linear_fwd: bad lora_dtype");
    hipStream_t stream = (hipStream_t)stream_;
    if (M == 0) return XQ_OK;
    XQ_REQUIRE(ldy % 8 == 0 && xq_aligned(y, 16), "xq_linear_fwd: y rows must be 16-byte aligned");
    const int rp = r_pad_of(r);
    // decode / rollout shapes: stream the packed weight once (HBM-bound kernel); forward only
    if (!su_out && takes_skinny(w, M, ldx, lora_A, lora_B, lora_dtype, r)) {
        rc = launch_skinny(w, (const bf16_t*)x, ldx, M, lora_A, lora_B, lora_dtype, r, scaling,
                           (const bf16_t*)bias_bf16, (bf16_t*)y, ldy, workspace, workspace_bytes, stream);
        if (rc != XQ_ERR_UNSUPPORTED) return rc;
    }
    bf16_t* su = nullptr;
    const LowRankRight right{{lora_B, nullptr}, r, r, rp, lora_dtype == XQ_DT_F32, 0};
    Carver cv{(workspace && xq_aligned(workspace, 256)) ? (uint8_t*)workspace : nullptr, 0, workspace_bytes};
    if (rp) {
        XQ_REQUIRE(workspace && xq_aligned(workspace, 256) && workspace_bytes >= linear_workspace_needed(M, N, K, r),
                   "xq_linear_fwd: workspace missing, misaligned or smaller than xq_linear_workspace_bytes()");
        su = su_out ? (bf16_t*)su_out : (bf16_t*)cv.take(M * rp * 2);
        bf16_t* panel = (bf16_t*)cv.take(lowrank_panel_bytes(1, M, rp, K));
        const LowRankJob job{(const bf16_t*)x, ldx, K, {lora_A, nullptr}, 1, r, rp, scaling, su, rp, 0};
        // (the sums of its splits live where the product's will)
        if ((rc = launch_lowrank(&job, 1, M, factor_mode(lora_dtype, false), panel, stream, (float*)cv.take(0), workspace_bytes - cv.used))) return rc;
    }
    // what is left of the workspace holds split-K partial sums (small row counts); without it the launch is unsplit
    float* partial = (float*)cv.take(0);
    return launch_tile_gemm(w, true, (const bf16_t*)x, ldx, M, nullptr, nullptr, su, nullptr, rp, (const bf16_t*)bias_bf16,
                            (bf16_t*)y, ldy, stream, "xq_linear_fwd", partial, partial ? workspace_bytes - cv.used : 0, nullptr,
                            rp ? &right : nullptr);
}

// ---- forward for callers that cannot allocate ------------------------------------------------------------------
// The scratch of xq_linear_fwd (prepared LoRA panels, the [M, r_pad] intermediate, split-K partial sums) in an
// array that is part of the loaded code object: each device the library runs on holds its own copy at its own
// address until the process ends.  Host code reaches it only through the address hipGetSymbolAddress returns with
// that device current; the array's name is a host-side handle, never a device address.
static __device__ __align__(256) unsigned char scratch[XQ_STATIC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

// device address of this device's copy of `scratch` (resolved once per device, with that device current)
static int static_scratch(void** out, const char* who) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        xq_set_error("%s: cannot identify the current device: %s", who, hipGetErrorString(e));
        return XQ_ERR_LAUNCH;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            xq_set_error("%s: hipGetSymbolAddress(scratch) failed on device %d: %s", who, dev, hipGetErrorString(e));
            return XQ_ERR_LAUNCH;
        }
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return XQ_OK;
}

extern "C" int64_t xq_static_scratch_bytes(void) { return XQ_STATIC_SCRATCH_BYTES; }

extern "C" int64_t xq_linear_fwd_swiglu_workspace_bytes_fmt(int format, int64_t M, int64_t N2, int64_t K, int r) {
    if (M < 0 || N2 < 0) return 0;
    return align256(xq_linear_workspace_bytes_fmt(format, M, N2, K, r)) + align256(M * N2 * 2) + 256;
}
extern "C" int64_t xq_linear_fwd_swiglu_workspace_bytes(int64_t M, int64_t N2, int64_t K, int r) {
    return xq_linear_fwd_swiglu_workspace_bytes_fmt(-1, M, N2, K, r);
}

extern "C" int xq_linear_fwd_swiglu(const xq_weight* w, const void* x, int64_t ldx, int64_t M, const void* lora_A, const void* lora_B,
                                    int lora_dtype, int r, float scaling, const void* bias_bf16, void* h, int64_t ldh, void* workspace,
                                    int64_t workspace_bytes, void* stream_) {
    int rc = check_dense(w, "xq_linear_fwd_swiglu");
    if (rc) return rc;
    const int64_t N2 = w->rows, K = w->cols, I = N2 / 2;
    XQ_REQUIRE(N2 % 16 == 0, "xq_linear_fwd_swiglu: the weight holds gate | up, [2 I, K] with I %% 8 == 0; got %lld rows", (long long)N2);
    XQ_REQUIRE(M >= 0 && (M == 0 || (x && h)), "xq_linear_fwd_swiglu: NULL activation pointer");
    XQ_REQUIRE(r >= 0 && r <= 64, "xq_linear_fwd_swiglu: LoRA rank %d out of range [0, 64]", r);
    XQ_REQUIRE(r == 0 || (lora_A && lora_B), "xq_linear_fwd_swiglu: LoRA factors are NULL");
    XQ_REQUIRE(lora_dtype == XQ_DT_F32 || lora_dtype == XQ_DT_BF16, "xq_linear_fwd_swiglu: bad lora_dtype");
    if (M == 0) return XQ_OK;
    XQ_REQUIRE(ldh % 8 == 0 && xq_aligned(h, 16), "xq_linear_fwd_swiglu: h rows must be 16-byte aligned");
    XQ_REQUIRE(workspace && xq_aligned(workspace, 256) && workspace_bytes >= xq_linear_fwd_swiglu_workspace_bytes_fmt(w->format, M, N2, K, r),
               "xq_linear_fwd_swiglu: workspace missing, misaligned or smaller than xq_linear_fwd_swiglu_workspace_bytes()");
    hipStream_t stream = (hipStream_t)stream_;
    // decode sizes: one launch that holds a column's gate and up rows in the same block
    if (g_skinny_enabled && skinny_rows_enabled() && skinny_supported(w, M) && ldx % 8 == 0 && ldx < (1ll << 31) && xq_aligned(x, 16) &&
        xq_aligned(w->packed, 16) && skinny_rows_swiglu_supported(w, M, lora_A, lora_B, lora_dtype, r)) {
        const double bytes = (double)xq_packed_bytes_per_expert(w) + (double)xq_scale_bytes_per_expert(w) + 2.0 * M * K + 2.0 * M * I +
                             4.0 * r * (K + N2);
        const bool timed = xq_profile_mark_begin(stream, bytes);
        rc = launch_skinny_rows_swiglu(w, (const bf16_t*)x, ldx, M, lora_A, lora_B, r, scaling, (const bf16_t*)bias_bf16, (bf16_t*)h, ldh,
                                       workspace, stream);
        if (rc != XQ_ERR_UNSUPPORTED) {      // (unsupported: no slot for the low-rank exchange could be had; nothing was launched)
            if (timed) xq_profile_mark_end(stream);
            if (rc) return rc;
            XQ_CHECK_LAUNCH("skinny forward with SwiGLU");
            return XQ_OK;
        }
    }
    // otherwise the forward into the workspace, then the elementwise kernel
    const int64_t lin = align256(xq_linear_workspace_bytes_fmt(w->format, M, N2, K, r));
    bf16_t* gu = (bf16_t*)((uint8_t*)workspace + lin);
    if ((rc = xq_linear_fwd(w, x, ldx, M, lora_A, lora_B, lora_dtype, r, scaling, bias_bf16, gu, N2, nullptr, workspace, lin, stream_))) return rc;
    return xq_silu_mul_fwd(gu, gu + I, N2, nullptr, h, ldh, M, I, stream_);
}

extern "C" int64_t xq_linear_fwd_multi_workspace_bytes(const xq_linear_job* jobs, int n_jobs, int64_t M) {
    int64_t need = 256 * 8, joint = 0;
    if (!jobs) return need;
    for (int i = 0; i < n_jobs; ++i) {
        if (!jobs[i].w) continue;
        const int64_t b = xq_linear_workspace_bytes_fmt(jobs[i].w->format, M, jobs[i].w->rows, jobs[i].w->cols, jobs[i].r);
        if (b > need) need = b;
        if (M <= 64) joint += skinny_workspace_bytes(M, jobs[i].w->rows, jobs[i].w->cols, r_pad_of(jobs[i].r));   // side by side in a joint launch
    }
    return need > joint ? need : joint;
}

extern "C" int xq_linear_fwd_multi(const xq_linear_job* jobs, int n_jobs, const void* x, int64_t ldx, int64_t M, int lora_dtype,
                                   void* workspace, int64_t workspace_bytes, void* stream_) {
    XQ_REQUIRE(jobs && n_jobs >= 1 && n_jobs <= XQ_LINEAR_MULTI_MAX, "xq_linear_fwd_multi: %d forwards (1 .. %d are taken)", n_jobs,
               XQ_LINEAR_MULTI_MAX);
    XQ_REQUIRE(lora_dtype == XQ_DT_F32 || lora_dtype == XQ_DT_BF16, "xq_linear_fwd_multi: bad lora_dtype");
    for (int i = 0; i < n_jobs; ++i) {
        XQ_REQUIRE(jobs[i].w, "xq_linear_fwd_multi: forward %d has no weight", i);
        int rc = check_dense(jobs[i].w, "xq_linear_fwd_multi");
        if (rc) return rc;
        XQ_REQUIRE(jobs[i].w->cols == jobs[0].w->cols, "xq_linear_fwd_multi: forward %d contracts over %lld features, forward 0 over %lld", i,
                   (long long)jobs[i].w->cols, (long long)jobs[0].w->cols);
        XQ_REQUIRE(jobs[i].r >= 0 && jobs[i].r <= 64, "xq_linear_fwd_multi: LoRA rank %d out of range [0, 64]", jobs[i].r);
        XQ_REQUIRE(jobs[i].r == 0 || (jobs[i].lora_A && jobs[i].lora_B), "xq_linear_fwd_multi: LoRA factors are NULL");
        XQ_REQUIRE(M == 0 || jobs[i].y, "xq_linear_fwd_multi: NULL output pointer");
        XQ_REQUIRE(M == 0 || (jobs[i].ldy % 8 == 0 && xq_aligned(jobs[i].y, 16)), "xq_linear_fwd_multi: y rows must be 16-byte aligned");
    }
    XQ_REQUIRE(M >= 0 && (M == 0 || x), "xq_linear_fwd_multi: NULL activation pointer");
    if (M == 0) return XQ_OK;
    hipStream_t stream = (hipStream_t)stream_;
    XQ_REQUIRE(workspace && xq_aligned(workspace, 256) && workspace_bytes >= xq_linear_fwd_multi_workspace_bytes(jobs, n_jobs, M),
               "xq_linear_fwd_multi: workspace missing, misaligned or smaller than xq_linear_fwd_multi_workspace_bytes()");
    // decode shapes that fit the whole-row kernel: every forward in one launch
    if (g_skinny_enabled && skinny_rows_enabled() && n_jobs > 1 && ldx % 8 == 0 && xq_aligned(x, 16)) {
        SkinnyRowsJob rj[XQ_LINEAR_MULTI_MAX];
        double bytes = 2.0 * M * jobs[0].w->cols;
        bool ok = true;
        for (int i = 0; i < n_jobs; ++i) {
            const xq_weight* w = jobs[i].w;
            rj[i] = SkinnyRowsJob{w, jobs[i].lora_A, jobs[i].lora_B, jobs[i].r, jobs[i].scaling, (const bf16_t*)jobs[i].bias_bf16,
                                  (bf16_t*)jobs[i].y, jobs[i].ldy};
            ok = ok && skinny_supported(w, M) && xq_aligned(w->packed, 16);
            bytes += (double)xq_packed_bytes_per_expert(w) + (double)xq_scale_bytes_per_expert(w) + 2.0 * M * w->rows +
                     4.0 * jobs[i].r * (w->cols + w->rows);
        }
        if (ok && skinny_rows_multi_supported(rj, n_jobs, M, lora_dtype)) {
            const bool timed = xq_profile_mark_begin(stream, bytes);
            const int rc = launch_skinny_rows_multi(rj, n_jobs, (const bf16_t*)x, ldx, M, workspace, stream);
            if (rc != XQ_ERR_UNSUPPORTED) {  // (unsupported: no slots for the low-rank exchange could be had; nothing was launched)
                if (timed) xq_profile_mark_end(stream);
                if (rc) return rc;
                XQ_CHECK_LAUNCH("skinny forwards");
                return XQ_OK;
            }
        }
    }
    // decode shapes outside the whole-row kernel: every forward in one streaming launch and one epilogue
    if (g_skinny_enabled && n_jobs > 1 && M <= 16 && ldx % 8 == 0 && xq_aligned(x, 16)) {
        SkinnyRowsJob sj[XQ_LINEAR_MULTI_MAX];
        double bytes = 2.0 * M * jobs[0].w->cols;
        bool ok = true;
        for (int i = 0; i < n_jobs; ++i) {
            const xq_weight* w = jobs[i].w;
            sj[i] = SkinnyRowsJob{w, jobs[i].lora_A, jobs[i].lora_B, jobs[i].r, jobs[i].scaling, (const bf16_t*)jobs[i].bias_bf16,
                                  (bf16_t*)jobs[i].y, jobs[i].ldy};
            ok = ok && skinny_takes_stream(w, M, ldx, jobs[i].lora_A, jobs[i].lora_B, lora_dtype, jobs[i].r);
            bytes += (double)xq_packed_bytes_per_expert(w) + (double)xq_scale_bytes_per_expert(w) + 2.0 * M * w->rows +
                     4.0 * jobs[i].r * (w->cols + w->rows);
        }
        if (ok && skinny_stream_multi_supported(sj, n_jobs, M)) {
            const bool timed = xq_profile_mark_begin(stream, bytes);
            const int rc = launch_skinny_stream(sj, n_jobs, false, (const bf16_t*)x, ldx, M, lora_dtype, workspace, stream);
            if (timed) xq_profile_mark_end(stream);
            if (rc) return rc;
            XQ_CHECK_LAUNCH("skinny forwards");
            return XQ_OK;
        }
    }
    // otherwise one after the other (the workspace is reused: the launches are ordered by the stream)
    for (int i = 0; i < n_jobs; ++i) {
        const int rc = xq_linear_fwd(jobs[i].w, x, ldx, M, jobs[i].lora_A, jobs[i].lora_B, lora_dtype, jobs[i].r, jobs[i].scaling,
                                     jobs[i].bias_bf16, jobs[i].y, jobs[i].ldy, nullptr, workspace, workspace_bytes, stream_);
        if (rc) return rc;
    }
    return XQ_OK;
}

extern "C" int xq_linear_fwd_static(const xq_weight* w, const void* x, int64_t ldx, int64_t M, const void* lora_A,
                                    const void* lora_B, int lora_dtype, int r, float scaling, const void* bias_bf16,
                                    void* y, int64_t ldy, void* stream_) {
    int rc = check_dense(w, "xq_linear_fwd_static");
    if (rc) return rc;
    XQ_REQUIRE(M >= 0, "xq_linear_fwd_static: negative row count");
    XQ_REQUIRE(r >= 0 && r <= 64, "xq_linear_fwd_static: LoRA rank %d out of range [0, 64]", r);
    const int64_t need = linear_workspace_needed(M, w->rows, w->cols, r);
    XQ_REQUIRE(need <= XQ_STATIC_SCRATCH_BYTES,
               "xq_linear_fwd_static: M=%lld, N=%lld, K=%lld, r=%d needs %lld bytes of scratch, the built-in buffer "
               "holds %lld; use xq_linear_fwd with a caller workspace",
               (long long)M, (long long)w->rows, (long long)w->cols, r, (long long)need,
               (long long)XQ_STATIC_SCRATCH_BYTES);
    void* ws = nullptr;
    if ((rc = static_scratch(&ws, "xq_linear_fwd_static"))) return rc;
    // nothing in the forward reads scratch it has not written in the same call (no counters, no accumulation into
    // memory), so the previous call's contents need no clearing
    return xq_linear_fwd(w, x, ldx, M, lora_A, lora_B, lora_dtype, r, scaling, bias_bf16, y, ldy, nullptr, ws,
                         XQ_STATIC_SCRATCH_BYTES, stream_);
}

extern "C" int xq_linear_bwd(const xq_weight* w, const void* x, int64_t ldx, const void* dy, int64_t lddy, int64_t M,
                             const void* lora_A, const void* lora_B, int lora_dtype, int r, float scaling,
                             const void* su_in, void* dx, int64_t lddx, float* dA, float* dB, void* workspace,
                             int64_t workspace_bytes, void* stream_) {
    int rc = check_dense(w, "xq_linear_bwd");
    if (rc) return rc;
    const int64_t N = w->rows, K = w->cols;
    XQ_REQUIRE(M >= 0 && (M == 0 || dy), "xq_linear_bwd: dy is NULL");
    XQ_REQUIRE(r >= 0 && r <= 64, "xq_linear_bwd: LoRA rank %d out of range [0, 64]", r);
    XQ_REQUIRE(r == 0 || (lora_A && lora_B), "xq_linear_bwd: LoRA factors are NULL");
    XQ_REQUIRE(lora_dtype == XQ_DT_F32 || lora_dtype == XQ_DT_BF16, "xq_linear_bwd: bad lora_dtype");
    XQ_REQUIRE(!(dA || dB) || r > 0, "xq_linear_bwd: factor gradients requested with r == 0");
    XQ_REQUIRE(!(dA || dB) || M == 0 || x, "xq_linear_bwd: x is needed for the factor gradients");
    hipStream_t stream = (hipStream_t)stream_;
    const int rp = r_pad_of(r);
    if (M == 0) {
        if (dA && (rc = launch_zero_fill(dA, (int64_t)r * K * 4, stream))) return rc;
        if (dB && (rc = launch_zero_fill(dB, N * r * 4, stream))) return rc;
        return XQ_OK;
    }
    bf16_t* v = nullptr;
    const bf16_t* su = (const bf16_t*)su_in;
    const LowRankRight right{{lora_A, nullptr}, K, r, rp, lora_dtype == XQ_DT_F32, 1};
    float* partial = nullptr;
    Carver cv{(workspace && xq_aligned(workspace, 256)) ? (uint8_t*)workspace : nullptr, 0, workspace_bytes};
    if (rp) {
        XQ_REQUIRE(workspace && xq_aligned(workspace, 256) && workspace_bytes >= linear_workspace_needed(M, N, K, r),
                   "xq_linear_bwd: workspace missing, misaligned or smaller than xq_linear_workspace_bytes()");
        v = (bf16_t*)cv.take(M * rp * 2);
        bf16_t* su_ws = (bf16_t*)cv.take(M * rp * 2);
        bf16_t* panel = (bf16_t*)cv.take(lowrank_panel_bytes(1, M, rp, K));
        // v = bf16(s * dy . B)   [M, rp]
        const LowRankJob jv{(const bf16_t*)dy, lddy, N, {lora_B, nullptr}, 1, r, rp, scaling, v, rp, 0};
        if ((rc = launch_lowrank(&jv, 1, M, factor_mode(lora_dtype, true), nullptr, stream, (float*)cv.take(0), workspace_bytes - cv.used))) return rc;
        if (dB && !su) {
            const LowRankJob ju{(const bf16_t*)x, ldx, K, {lora_A, nullptr}, 1, r, rp, scaling, su_ws, rp, 0};
            if ((rc = launch_lowrank(&ju, 1, M, factor_mode(lora_dtype, false), panel, stream, (float*)cv.take(0), workspace_bytes - cv.used))) return rc;
            su = su_ws;
        }
    }
    // one region after the carved buffers: split-K partial sums of the dgrad first, then (stream order) the
    // partial sums of the factor gradients
    partial = (float*)cv.take(0);
    if (dx) {
        XQ_REQUIRE(lddx % 8 == 0 && xq_aligned(dx, 16), "xq_linear_bwd: dx rows must be 16-byte aligned");
        if ((rc = launch_tile_gemm(w, false, (const bf16_t*)dy, lddy, M, nullptr, nullptr, v, nullptr, rp, nullptr, (bf16_t*)dx,
                                   lddx, stream, "xq_linear_bwd(dx)", partial, partial ? workspace_bytes - cv.used : 0, nullptr,
                                   rp ? &right : nullptr)))
            return rc;
    }
    // dB[N, r] = dy^T . su ; dA[r, K] = (x^T . v)^T
    TnJob jobs[2];
    int n = 0;
    if (dB) jobs[n++] = TnJob{(const bf16_t*)dy, lddy, N, su, rp, rp, r, false, dB};
    if (dA) jobs[n++] = TnJob{(const bf16_t*)x, ldx, K, v, rp, rp, r, true, dA};
    return n ? launch_tn_multi(jobs, n, M, partial, stream) : XQ_OK;
}

extern "C" int xq_grouped_gemm(const xq_weight* w, int transpose_w, const void* a, int64_t lda, int64_t n_rows,
                               const int32_t* offsets, const int32_t* tile_offsets, const void* su,
                               const void* lora_right, int r_pad, void* y, int64_t ldy, void* stream) {
    int rc = xq_validate_weight(w, "xq_grouped_gemm");
    if (rc) return rc;
    XQ_REQUIRE(offsets && tile_offsets, "xq_grouped_gemm: offsets / tile_offsets are NULL");
    XQ_REQUIRE(n_rows == 0 || (a && y), "xq_grouped_gemm: NULL activation pointer");
    XQ_REQUIRE(ldy % 8 == 0 && xq_aligned(y, 16), "xq_grouped_gemm: y rows must be 16-byte aligned");
    // bank is [E, K_in, N_out]: forward contracts over W rows, dgrad over W cols
    return launch_tile_gemm(w, transpose_w != 0, (const bf16_t*)a, lda, n_rows, offsets, tile_offsets, (const bf16_t*)su,
                            (const bf16_t*)lora_right, r_pad, nullptr, (bf16_t*)y, ldy, (hipStream_t)stream,
                            "xq_grouped_gemm", nullptr, 0);
}

extern "C" int xq_factor_prep(const void* in, int in_dtype, int64_t rows_in, int64_t cols_in, int transpose,
                              void* out_bf16, int64_t rows_out, int64_t cols_out, int64_t num_experts, void* stream) {
    XQ_REQUIRE(in_dtype == XQ_DT_F32 || in_dtype == XQ_DT_BF16, "xq_factor_prep: bad dtype");
    XQ_REQUIRE(num_experts == 0 || rows_out * cols_out == 0 || (in && out_bf16), "xq_factor_prep: NULL pointer");
    int64_t need_r = transpose ? cols_in : rows_in, need_c = transpose ? rows_in : cols_in;
    XQ_REQUIRE(rows_out >= need_r && cols_out >= need_c, "xq_factor_prep: output [%lld, %lld] smaller than source", (long long)rows_out, (long long)cols_out);
    return launch_factor_prep(in, in_dtype, rows_in, cols_in, transpose != 0, (bf16_t*)out_bf16, rows_out, cols_out,
                              num_experts, (hipStream_t)stream);
}

extern "C" int xq_grouped_lora_down(const void* a, int64_t lda, int64_t n_rows, const int32_t* offsets,
                                    const int32_t* tile_offsets, int32_t num_experts, const void* F, int shared,
                                    int r_pad, int64_t K, float scale, void* t, void* stream) {
    XQ_REQUIRE(offsets && tile_offsets && num_experts >= 1, "xq_grouped_lora_down: offsets / tile_offsets are NULL");
    XQ_REQUIRE(n_rows == 0 || (a && F && t), "xq_grouped_lora_down: NULL pointer");
    return launch_small_nt((const bf16_t*)a, lda, n_rows, K, (const bf16_t*)F, r_pad, scale, (bf16_t*)t, offsets,
                           tile_offsets, num_experts, shared != 0, (hipStream_t)stream);
}

extern "C" int64_t xq_lora_wgrad_workspace_bytes(int64_t n_rows, int64_t width, int r_pad) {
    return tn_partial_bytes(n_rows, width, r_pad) + 256;
}

extern "C" int xq_grouped_lora_wgrad(const void* P, int64_t ldp, int64_t p_width, const void* Q, int r_pad, int r_out,
                                     int64_t n_rows, const int32_t* offsets, int32_t num_experts, int transpose_out,
                                     float* out, void* workspace, const int32_t* row_limit, void* stream) {
    XQ_REQUIRE(out && (n_rows == 0 || (P && Q)), "xq_grouped_lora_wgrad: NULL pointer");
    if (n_rows == 0 && !offsets) return launch_zero_fill(out, p_width * r_out * 4, (hipStream_t)stream);
    return launch_tn((const bf16_t*)P, ldp, p_width, (const bf16_t*)Q, r_pad, r_out, n_rows, transpose_out != 0, out,
                     (float*)workspace, offsets, num_experts, (hipStream_t)stream, row_limit);
}
