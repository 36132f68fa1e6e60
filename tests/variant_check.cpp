// The rules that pick each shape's kernel variants (csrc/variants.hpp), for
// every power-of-two N up to 2^24 and every limb count up to 300, with the
// shape fields of the plan, prime counts at both ends of a limb count's range,
// every split n1, and tile counts from one to all: the variant that a rule
// names is one that is compiled.  Plans outside the lists are told apart.
// Prints "ok <shapes>", or with arguments <N> <limbs> <primes> the variants of
// that product, all tiles at once.
#include <cstdio>
#include <cstdlib>

#include "variants.hpp"

static pm::Shape shape(uint32_t n, uint32_t limbs, uint32_t r, uint32_t n1) {
    pm::Shape s;
    s.n = n, s.limbs = limbs, s.r = r, s.n1 = n1, s.n2 = n / n1;
    s.n_pad = (n + 255) / 256 * 256;
    s.r_pad = (r + 63) / 64 * 64;
    s.conv_k = (4 * limbs + 63) / 64 * 64;
    s.conv_rows = 4 * s.r_pad;
    s.crt_words = limbs + 4;
    s.crt_words_pad = (s.crt_words + 63) / 64 * 64;
    s.crt_rows = 4 * s.crt_words_pad;
    s.t_words = limbs + 2;
    s.row_width = n < 2048 ? n : 2048;
    if (s.row_width < n1) s.row_width = n1;
    s.rows = n / s.row_width;
    return s;
}

static void print(const pm::Shape& s) {
    const uint32_t tiles = s.n_pad / pm::kTile, logc = pm::row_variant(s.row_width, s.n1);
    const pm::TileSet all = pm::tile_range(0, tiles);
    if (pm::conversion_short(s)) {
        const pm::ConvertPlan p = pm::convert_plan(s, 2 * tiles, pm::kConvertBlocks, pm::conversion_columns(s, all));
        std::printf("convert<%u,%u,%u>\n", p.ks, p.nt, p.rows);
    } else {
        const uint64_t blocks = uint64_t(s.conv_rows / pm::kTile) * 2 * tiles;
        std::printf("conversion_gemm<%d> %llu\n", pm::gemm_halves(blocks) ? 1 : 2, (unsigned long long)blocks);
    }
    if (logc) std::printf("ntt_rows_reg<%u,%u>\n", logc, s.n1);
    else std::printf("ntt_rows_product\n");
    if (pm::reconstruct_fused(s)) {
        std::printf("crt_reconstruct<%u>\n", pm::fused_waves(s.crt_words));
        return;
    }
    const uint64_t blocks = uint64_t(s.crt_rows / pm::kTile) * tiles;
    if (pm::crt_few_blocks(s.crt_rows, tiles)) std::printf("crt_small %u\n", (s.r + 15) / 16);
    else std::printf("crt_gemm<%d> %llu\n", pm::gemm_halves(blocks) ? 1 : 2, (unsigned long long)blocks);
    const pm::Reconstruction v = pm::reconstruct_variant(s, tiles);
    std::printf("%s\n", v == pm::Reconstruction::kWave      ? "reconstruct_waves"
                        : v == pm::Reconstruction::kLanes32 ? "reconstruct_wide<32>"
                                                            : "reconstruct_wide<64>");
}

int main(int argc, char** argv) {
    if (argc == 4) {
        print(shape(std::atoi(argv[1]), std::atoi(argv[2]), std::atoi(argv[3]), 1));
        return 0;
    }
    unsigned long shapes = 0;
    for (uint32_t log_n = 0; log_n <= 24; ++log_n)
        for (uint32_t limbs = 1; limbs <= 300; ++limbs)
            for (uint32_t n1 = 1; n1 <= 2048 && n1 <= (1u << log_n); n1 *= 2)
                // primes of 30 to 31 bits cover 4N (q-1)^2, q of 1 bit to all of the limbs
                for (uint32_t r : {1u, 64 * limbs / 31 + 1, (64 * limbs + log_n + 2) / 30 + 1}) {
                    const pm::Shape s = shape(1u << log_n, limbs, r, n1);
                    const uint32_t tiles = s.n_pad / pm::kTile, logc = pm::row_variant(s.row_width, s.n1);
                    auto fail = [&](const char* what, const pm::ConvertPlan& p) {
                        std::printf("%s: N=%u L=%u r=%u n1=%u <%u,%u,%u>\n", what, s.n, limbs, r, n1, p.ks, p.nt, p.rows);
                        std::exit(1);
                    };
                    ++shapes;
                    if (logc && !pm::rows_compiled(logc, s.n1)) fail("rows", {});
                    if (s.row_width % 256 == 0 && s.rows <= 64 && !pm::columns_compiled(s.rows)) fail("columns", {});
                    if (!pm::conversion_short(s)) continue;
                    const bool columns = pm::conversion_columns(s, pm::tile_range(0, tiles));
                    for (uint32_t nops = 1; nops <= 2; ++nops) {
                        for (uint32_t t = 1; t < tiles; t *= 2) {
                            const pm::ConvertPlan p = pm::convert_plan(s, nops * t, pm::kConvertBlocks, false);
                            if (!pm::convert_compiled(p) || !p.split) fail("some tiles", p);
                        }
                        const pm::ConvertPlan p = pm::convert_plan(s, nops * tiles, pm::kConvertBlocks, columns);
                        if (!pm::convert_compiled(p) || !p.split) fail("all tiles", p);
                        // a lane holds whole columns of the [rows][2048] matrix
                        if (columns && (p.rows != s.rows || s.row_width != 2048 || p.nt % p.rows)) fail("whole columns", p);
                    }
                    if (limbs > pm::kGroupShortLimbs) continue;
                    const pm::ConvertPlan p = pm::convert_plan(s, 2 * tiles, pm::kConvertGroupBlocks, true);
                    if (!pm::convert_group_compiled(p)) fail("batch", p);
                    // a batch's product: spread over the GPU where it is alone,
                    // kConvertGroupBlocks or what one split gives among many
                    const uint32_t chunks = (r + 15) / 16, blocks = pm::convert_group_blocks(s.n, p.nt);
                    const uint32_t alone = pm::convert_group_split(chunks, blocks, blocks);
                    const uint32_t among = pm::convert_group_split(chunks, blocks, 1 << 20);
                    if (blocks > 2 * tiles * (pm::kTile / (64 * p.nt))) fail("batch blocks", p);
                    if (alone < 1 || alone > chunks || (alone < chunks && blocks * alone < pm::kConvertBlocks))
                        fail("alone in a batch", p);
                    if (among < 1 || among > alone || (among > 1 && blocks * (among - 1) >= pm::kConvertGroupBlocks))
                        fail("among many in a batch", p);
                }
    // variants that no rule may name
    for (pm::ConvertPlan p : {pm::ConvertPlan{3, 4, 1, 1}, pm::ConvertPlan{16, 2, 4, 1}, pm::ConvertPlan{8, 8, 8, 1}})
        if (pm::convert_compiled(p) || pm::convert_group_compiled(p)) return std::printf("foreign convert variant\n"), 1;
    if (pm::convert_group_compiled({16, 2, 1, 1}) || pm::rows_compiled(6, 1) || pm::rows_compiled(11, 16) ||
        pm::columns_compiled(0) || pm::columns_compiled(3) || pm::columns_compiled(128))
        return std::printf("foreign variant\n"), 1;
    std::printf("ok %lu\n", shapes);
    return 0;
}
