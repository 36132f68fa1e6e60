// Which kernel variant each shape takes (no HIP dependence, so the CPU tests
// include it directly): the rules of the launch wrappers in kernels.hip, and the
// lists of the variants that are compiled.
#pragma once

#include <cstdint>

#include "chunks.hpp"
#include "plan.hpp"

namespace pm {

constexpr uint32_t kTile = 256;  // coefficients, or weight rows, of a whole GEMM tile
constexpr uint32_t kTK = 64;     // bytes of K per step

// ---- conversion ---------------------------------------------------------

// Packing and conversion in one kernel that reads a and b itself (launch_convert),
// for q of up to kShortLimbs limbs.
constexpr uint32_t kShortLimbs = 256;
inline bool conversion_short(const Shape& s) { return s.limbs <= kShortLimbs; }

// Variant of the short conversion: K steps held in registers (KS), 16-coefficient
// fragments per wave (NT), transform rows whose column stages a lane does (1:
// none), splits of the primes over blocks.
struct ConvertPlan {
    uint32_t ks, nt, rows, split;
};
#define PM_CONVERT_VARIANTS(X)                                                                         \
    X(1, 1, 1) X(2, 1, 1) X(4, 1, 1) X(8, 1, 1) X(16, 1, 1) X(1, 4, 1) X(2, 4, 1) X(4, 4, 1) X(8, 2, 1) \
        X(16, 2, 1) X(1, 4, 2) X(2, 4, 2) X(4, 4, 2) X(8, 2, 2) X(16, 2, 2) X(1, 4, 4) X(2, 4, 4)       \
            X(4, 4, 4) X(8, 4, 4) X(1, 8, 8) X(2, 8, 8)
// Those of a batch's one kernel (convert_group), which picks among them itself.
#define PM_CONVERT_GROUP_VARIANTS(X)                                                                   \
    X(1, 4, 1) X(2, 4, 1) X(4, 4, 1) X(8, 2, 1) X(1, 4, 2) X(2, 4, 2) X(4, 4, 2) X(8, 2, 2) X(1, 4, 4) \
        X(2, 4, 4) X(4, 4, 4)

constexpr uint32_t kConvertBlocks = 512, kConvertGroupBlocks = 64;  // two per CU; a batch's share at least
// Up to here a batch's products take the short conversion: 16 K steps in
// registers would cost the shared kernel a third of its occupancy.
constexpr uint32_t kGroupShortLimbs = 128;

// `tiles` 256-coefficient tiles in all (of both operands).  Wide waves (NT 2 or
// 4) read each weight from LDS for 32 or 64 coefficients; where they would
// leave most of the GPU idle (fewer than want_blocks / 2 blocks even with every
// 16 primes in a block of their own) waves of 16 coefficients take over: N =
// 1024 with 8 limbs 3.5 us against 4.3 with 64-coefficient blocks.  Then the
// primes are split until there are want_blocks blocks.  In a batch the waves are
// wide, and convert_group_split splits the primes.
//
// `columns`: a lane takes the column stages where it holds whole columns, with
// as many rows as fragments at most (8 with up to two K steps, 4 with up to
// eight are what the registers hold; a batch, whose one kernel has three waves
// per SIMD, keeps the wide waves' own).
// That saves a pass over the residues and a launch, and is worth wide waves at
// any number of blocks, whole products in us: N = 4096 with 1 limb 28.3 -> 25.8,
// with 32 limbs 38.6 -> 36.0, with 125 65.9 -> 61.3, with 256 96.6 -> 89.4; N =
// 8192 with 2 limbs 28.5 -> 26.3, with 64 64.7 -> 59.7, with 128 94.0 -> 90.9;
// N = 16384 with 2 limbs 29.2 -> 28.4, with 28 44.1 -> 41.7.
inline ConvertPlan convert_plan(const Shape& s, uint32_t tiles, uint32_t want_blocks, bool columns) {
    const uint32_t ksteps = s.conv_k / kTK, chunks = (s.r + 15) / 16;
    const uint32_t ks = ksteps <= 1 ? 1 : ksteps <= 2 ? 2 : ksteps <= 4 ? 4 : ksteps <= 8 ? 8 : 16;
    const bool batch = want_blocks == kConvertGroupBlocks;
    const uint32_t wide = ks >= 8 ? 2 : 4, most = batch ? wide : ks <= 2 ? 8 : ks <= 8 ? 4 : 2;
    const uint32_t rows = columns && s.rows <= most ? s.rows : 1;
    uint32_t nt = rows > wide ? rows : wide;
    if (rows == 1 && !batch && tiles * 4 / nt * chunks < want_blocks / 2) nt = 1;
    const uint32_t blocks = tiles * 4 / nt, want = (want_blocks + blocks - 1) / blocks;
    return ConvertPlan{ks, nt, rows, chunks < want ? chunks : want};
}

// Splits of a batch product's primes, from its blocks without splits (the ones
// that hold coefficients) and those of all the batch's products.  Where the
// others fill the GPU a product needs no more than kConvertGroupBlocks: the batch
// of 64 small products' conversions took 152 us in all (in four launches then),
// and 210 with each product spread as if it were alone.  A few products do not
// fill it and are spread as far as one alone, in us (in brackets: split for
// kConvertGroupBlocks each): one of N = 4096 with 128 limbs 18.0 (43.0), two of
// N = 2048 16.3 (25.6), one of N = 2048 with 100 limbs 9.7 (18.8).  Twice
// kConvertBlocks was up to 4 % slower (8 products of N = 2048 with 128 limbs) and
// nowhere faster by more than runs differ.
inline uint32_t convert_group_split(uint32_t chunks, uint32_t blocks, uint64_t batch_blocks) {
    const uint64_t own = (kConvertGroupBlocks + blocks - 1) / blocks;
    const uint64_t fill = (kConvertBlocks + batch_blocks - 1) / batch_blocks;
    const uint64_t want = own > fill ? own : fill;
    return uint32_t(want < chunks ? want : chunks);
}
inline uint32_t convert_group_blocks(uint32_t n, uint32_t nt) { return 2 * ((n + 64 * nt - 1) / (64 * nt)); }

// Whether the short conversion of the tiles of `ts` takes the forward column
// stages too: every tile at once, and two to eight transform rows, fewer for
// wider q.
inline bool conversion_columns(const Shape& s, const TileSet& ts) {
    if (!conversion_short(s) || ts.t0 != 0 || ts.w != ts.count || ts.count != s.n_pad / kTile) return false;
    return convert_plan(s, ts.count, kConvertBlocks, true).rows > 1;
}

// ---- transform rows -----------------------------------------------------

// log2 of the row width the register kernel takes, or 0 where the LDS kernel
// runs: rows narrower than 128 values, and blocks wider than 8.
inline uint32_t row_variant(uint32_t row_width, uint32_t n1) {
    uint32_t logc = 0;
    while ((1u << logc) < row_width) ++logc;
    return logc >= 7 && n1 <= 8 ? logc : 0;
}
#define PM_ROWS_VARIANTS(X)                                                                                 \
    X(7, 1) X(7, 2) X(7, 4) X(7, 8) X(8, 1) X(8, 2) X(8, 4) X(8, 8) X(9, 1) X(9, 2) X(9, 4) X(9, 8) X(10, 1) \
        X(10, 2) X(10, 4) X(10, 8) X(11, 1) X(11, 2) X(11, 4) X(11, 8)

// ---- GEMM tiles ---------------------------------------------------------

// Whether a GEMM of `blocks` whole tiles takes halves (WN = 1).  A CU holds one
// whole tile's block, or two halves, at a time; halves pay when they spread what
// is left for the last round (up to 128 tiles on 256 CUs) over twice the CUs.
// CRT GEMM, whole against halves: 128 tiles 31.7 / 22.1 us (N = 8192, 226
// limbs), 80 tiles 62 / 42, 112 tiles 177 / 117 (N = 1024, 1747 limbs), but 224
// tiles 202 / 219 and 256 tiles 36.2 / 37.5; conversion GEMM 336 tiles 66 / 55,
// 456 tiles 190 / 195, 512 tiles 36.1 / 35.2.  With two full rounds and more the
// last one matters less than the halves' extra weight traffic.
inline bool gemm_halves(uint64_t blocks) { return blocks < 512 && (blocks - 1) % 256 < 128; }

// Whether the CRT GEMM has so few whole tiles that crt_small takes it.  Against
// halves: 3 tiles 6.4 / 13 us (N = 128, 128 limbs), 8 tiles 12.9 / 30.3 (N =
// 128, 500 limbs), 32 tiles 13.9 / 18.4 (N = 2048, 226 limbs), 28 tiles 68 / 98
// (N = 128, 1747 limbs); 80 tiles 63.6 / 41.8, where every wave reading its own
// operands from L2 starts to bound it.
inline bool crt_few_blocks(uint32_t crt_rows, uint32_t tiles) { return crt_rows / kTile * tiles < 48; }

// ---- CRT and reconstruction ---------------------------------------------

// Up to 60 limbs (64 word sums) one kernel does the CRT GEMM and the
// reconstruction, and the sums stay in LDS; wider q takes the GEMM, then a
// reconstruction from the sums in memory (reconstruct_variant).
constexpr uint32_t kFusedWords = 64;
inline bool reconstruct_fused(const Shape& s) { return s.crt_words <= kFusedWords; }
// Up to 8 transform rows, and the whole product at once: the fused kernel reads
// the row stage's results itself and does the inverse column stages (with one
// row: none) on their way into its operand layout in LDS.
inline bool residues_from_planes(const Shape& s, const TileSet& ts) {
    return s.rows <= 8 && reconstruct_fused(s) && (s.rows == 1 || (ts.t0 == 0 && ts.w == ts.count && ts.count == s.n_pad / kTile));
}
// Wave rows of the fused kernel: 16 word sums each.
constexpr uint32_t fused_waves(uint32_t crt_words) { return crt_words <= 16 ? 1 : crt_words <= 32 ? 2 : 4; }

// Reconstruction from the word sums: 32 or 64 lanes per coefficient with four
// words each (reconstruct_wide), or a wave with 64 words a round.
enum class Reconstruction { kLanes32, kLanes64, kWave };
constexpr uint32_t kWideWords = 256;
inline Reconstruction reconstruct_variant(const Shape& s, uint32_t tiles) {
    if (s.crt_words > kWideWords) return Reconstruction::kWave;
    // Up to 8 tiles leave the GPU idle, and the shorter path counts.  That is a
    // wave each where q's limbs fill whole rounds of 64 words (the round with
    // q's top words then has no empty words to carry a borrow through), whole
    // products at N = 128 and 2048 in us, wave against lanes: 64 limbs 30.9 /
    // 31.2 and 35.6 / 35.6, 127 limbs 1.6 and 1.3 shorter, 128 limbs 33.9 / 35.4
    // and 48.6 / 50.0, 192 limbs 0.8 and 0.7 shorter.  Elsewhere the lanes are:
    // 61 limbs 32.6 / 31.1 and 36.2 / 34.2, 100 limbs 33.9 / 32.3 and 41.3 / 39.5,
    // 160 limbs 37.7 / 37.0 and 56.3 / 55.4, 252 limbs 39.9 / 39.2 and 67.3 / 66.1.
    if (tiles <= 8 && (s.limbs + 1) % 64 <= 1) return Reconstruction::kWave;
    return s.crt_words <= 128 ? Reconstruction::kLanes32 : Reconstruction::kLanes64;
}

// ---- the compiled variants ----------------------------------------------

// A shape whose rule names a variant that is not compiled must fail, not leave
// its buffers unwritten: the launch wrappers throw where these say false.
inline bool convert_compiled(const ConvertPlan& cp) {
#define PM_IS(K, N, R) || (cp.ks == K && cp.nt == N && cp.rows == R)
    return false PM_CONVERT_VARIANTS(PM_IS);
}
inline bool convert_group_compiled(const ConvertPlan& cp) {
    return false PM_CONVERT_GROUP_VARIANTS(PM_IS);
#undef PM_IS
}
inline bool rows_compiled(uint32_t logc, uint32_t n1) {
#define PM_IS(LC, B) || (logc == LC && n1 == B)
    return false PM_ROWS_VARIANTS(PM_IS);
#undef PM_IS
}
// Row counts of the register column kernels: forward from 2, inverse from 1.
inline bool columns_compiled(uint32_t rows) { return rows >= 1 && rows <= 64 && (rows & (rows - 1)) == 0; }

}  // namespace pm
