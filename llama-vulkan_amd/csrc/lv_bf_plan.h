// lv_bf_plan.h — tiles, K slices and orders of bfloat16 products of many tokens (lv_bf16_gemm.h), by their sizes.
//
// Time = rounds of workgroups over 256 CUs x K steps x a step's time, plus prologue and epilogue, plus writing and reading a slice more.
// Fitted to launches whose weights come from HBM, as a model's do (with weights in the infinity cache wide tiles look better than they
// are), 1230 of them, 512 to 8192 columns and 16 to 2048 tokens, of which the choice is 1.1 % slower than the fastest in the mean; and to 230
// whole prompts of 13 models 1024 to 8192 wide, a product's tiles changed at a time: 0.6 % slower.  us,
// 128 x 128 tiles and 256 rows x 128, 160, 192 and 256 tokens; few workgroups take as long a step as they load:
//   100 tokens x 5248 x 5120 72 86 88 88 119; 128 x 3200 x 3072 45 47 48 48 73; 100 x 2048 x 2048 31 35, x 3072 x 768 15 21, x 4096 x 512 12 16;
//   16 x 8848 x 2048 29 25 26 26 46; 100 x 8848 x 2048 32 35 35 35 52; 300 x 22016 x 4096 109 89 78 69 95; 500 x 18560 x 4096 135 124 135 80 108;
//   777 x 22016 x 4096 193 159 148 145 191; 777 x 18560 x 4096 144 126 157 155 209; 777 x 2112 x 4096 57 53 76 72 101; 777 x 4096 x 11008 in two
//   slices 93 82 109 96 137, in three 124 106 82 79 101; 1000 x 8848 x 2048 63 66 45 46 62; 1100 x 18560 x 4096 204 187 168 174 210;
//   1900 x 22016 x 4096 346 328 335 324 294; 2048 x 13600 x 4096 279 250 234 244 217; 2048 x 4096 x 8192 144 123 133 130 187.
#pragma once

#include <cmath>
#include <cstdint>

namespace lv {

constexpr int kBfTile = 128;       // tokens per workgroup, bf16
constexpr int kBfStep = 64;

enum class BfTiles { k128, kWide, kWide160, kWide192, kWidest };

constexpr double kBfCus = 256, kBfEnds = 8, kBfWideEnds = 4;      // us before the first step and behind the last one; wide tiles': more
struct BfOffer {
    BfTiles tiles;
    uint32_t tokens;
    double busy, idle;      // us of a step, every CU at work and few of them
};
constexpr BfOffer kBfOffers[] = {{BfTiles::kWide, 128, 0.87, 0.76}, {BfTiles::kWide160, 160, 1.12, 0.87}, {BfTiles::kWide192, 192, 1.24, 0.88}, {BfTiles::kWidest, 256, 1.54, 1.27}};

// us of a K step of all rounds
inline double bf_small_step(double tiles)      // two share a CU
{
    const double left = std::fmod(tiles, 2 * kBfCus);
    return std::floor(tiles / (2 * kBfCus)) * 1.2 + (left > kBfCus ? 0.91 + 0.13 * left / kBfCus : left > 0 ? 0.76 : 0.0);
}
inline double bf_wide_step(const BfOffer &o, double tiles)
{
    const double last = std::fmod(tiles, kBfCus);
    return std::floor(tiles / kBfCus) * o.busy + (last > 0 ? o.idle + (o.busy - o.idle) * last / kBfCus : 0.0);
}
// of a tile that holds a part of its tokens: what its loads take whatever their number, and its products
inline double bf_part(double share) { return 0.57 + 0.43 * share; }

struct BfPlan {
    BfTiles tiles;
    uint32_t slices;
};
// a product of n tokens, cut into `slices` slices of K at most (the reader of the result adds them up)
inline BfPlan bf_plan(uint32_t rows, uint32_t n, uint32_t kp, uint32_t slices)
{
    BfPlan best{BfTiles::k128, 1};
    double best_us = 1e30;
    for (uint32_t s = 1; s <= slices; s++) {
        const uint32_t steps = (kp / kBfStep + s - 1) / s;
        if (s > 1 && steps < 8) break;
        // a slice more is written and read again, from the L2s while all of them fit there
        const double more = kBfEnds + (s - 1) * (1.0 + ((uint64_t)s * n * rows * 4 < 32u << 20 ? 1e-6 : 2e-6) * n * rows);
        auto take = [&](BfTiles t, double us) {
            if (us < best_us) {
                best_us = us;
                best = {t, s};
            }
        };
        take(BfTiles::k128, bf_small_step((double)((rows + 127) / 128) * ((n + 127) / 128) * s) * steps + more);
        for (const BfOffer &o : kBfOffers) {
            const uint32_t whole = n / o.tokens, rest = n % o.tokens, token_tiles = whole + (rest != 0);
            const double part = !rest ? 0.0 : o.tiles == BfTiles::kWidest ? 1.0 : bf_part((rest + 31) / 32 * 32.0 / o.tokens);
            const double us = bf_wide_step(o, (double)((rows + 255) / 256) * token_tiles * s) * (whole + part) / token_tiles * steps + kBfWideEnds + more;
            // 160 and 192 tokens, slices of long rows: up to 1.6 times the estimate (460 x 7168 x 19392, 160 in three 240, 128 in two 149), so only
            // where they gain more than a little
            take(o.tiles, s > 1 && (o.tokens == 160 || o.tokens == 192) ? 1.04 * us : us);
        }
    }
    return best;
}

// Tokens of an expert's tiles, 128 or 160, and their order.  us of gate and up, and of down (64 experts, 8 a token, 2048 x 4096 and
// 4096 x 1024): tiles of 128, a row tile after the other, then an expert after the other; tiles of 160 likewise.
//    300 tokens            239 180 241 179   127 121 127 121
//    900                   273 240 265 199   168 170 166 161
//   1400                   280 250 327 310   227 198 228 221
//   2048                   372 356 329 309   259 281 270 242
//    600, unevenly chosen  226 214 226 219   136 142 133 148
//   2048, unevenly chosen  356 364 344 372   272 282 257 279
// Few tokens an expert: the weights' way from HBM counts, an expert after the other; 160 where an expert of the mean number of choices
// and two standard deviations more then has fewer tiles, and where every round of workgroups is not one of few (32 experts, 4 a token, 2048
// x 2048 and 2048 x 1024, 900 tokens: 128 85 and 52, 160 92 and 62).  Down of 48 tokens an expert and more in tiles of 128: its weights are half
// as many and uneven experts decide (512 tokens of a prompt, unevenly chosen: 135 and 146).  Many: runs of one length whoever is chosen.
struct ExpertPlan {
    uint32_t tile;
    bool by_expert, down_by_expert;
};
inline ExpertPlan expert_plan(uint32_t n, uint32_t top, uint32_t experts, uint32_t rows)
{
    const double mean = (double)n * top / experts, many = mean + 2 * std::sqrt(mean);
    if (mean >= 192) return {160, false, false};
    const bool longer = experts * ((rows + 255) / 256) >= 512 && std::ceil(many / 160) < std::ceil(many / 128);
    return {longer ? 160u : 128u, true, longer || mean < 48};
}

}  // namespace lv
