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

// 128 tokens, one round, half of them or fewer in the rest: its tile is done with a step sooner, runs ahead and brings the weights of its rows to
// the L2 for the other tiles (5248 rows x 5120: 512 and 640 tokens 84 us, 900, seven tiles and four tokens, 72; measured from 512 rows on)
constexpr double kBfAhead = 0.67;

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
            const double tiles = (double)((rows + 255) / 256) * token_tiles * s;
            double step_us = bf_wide_step(o, tiles) * (whole + part) / token_tiles;
            if (o.tiles == BfTiles::kWide && tiles <= kBfCus && whole && rest && rest <= 64 && rows >= 512) step_us = std::fmin(step_us, kBfAhead + 0.5 * (o.busy - kBfAhead) * tiles / kBfCus);
            const double us = step_us * steps + kBfWideEnds + more;
            // 160 and 192 tokens, slices of long rows: up to 1.6 times the estimate (460 x 7168 x 19392, 160 in three 240, 128 in two 149), so only
            // where they gain more than a little
            take(o.tiles, s > 1 && (o.tokens == 160 || o.tokens == 192) ? 1.04 * us : us);
        }
    }
    return best;
}

// A layer's two products of chosen experts, over tiles of at most kBfTile tokens, an expert's each: 128 x 128 or 256 rows x 128
struct ExpertPlan {
    BfTiles gate_up, down;
    bool gate_up_by_expert;      // an expert after the other, not a row tile after the other
};
struct ExpertShape {
    uint32_t experts, top, rows, kp, down_rows, down_kp;      // rows: of an expert's gate and up
};
// How many tiles an expert has: choices spread about their mean as a normal variable, a little wider than even chances make them
inline double expert_tiles(double mean, uint32_t tile)
{
    const double spread = std::sqrt(2 * (mean + 0.03 * mean * mean));
    double tiles = 1 - std::exp(-mean);
    for (uint32_t k = 1; k < 4096; k++) {
        const double p = 0.5 * std::erfc((k * (double)tile + 0.5 - mean) / spread);
        if (p < 1e-3) break;
        tiles += p;
    }
    return tiles;
}
// By the estimate of bf_plan, the ends of wide tiles longer still: an expert's rows are gathered, and its tiles end at other times than others'.
// Us a layer in prompts of models of several layers (experts, a token's, feed-forward x width, tokens), 256 rows x 128, a row tile after the other,
// and what is more or less with: gate and up an expert after the other; 128 x 128 tiles of gate and up, of down; 256 rows x 160 tokens
//   8, 2, 512 x 1024       100  155    -0   -2  -5    +1      512  197   -0   -2   -5   +11     1600  339    0   -2   -5   +11
//   16, 4, 512 x 512       100  139    -1   -4  -5     0      512  174    0   -3   -5    +9     1600  292    0   -2   -4    +9
//   64, 8, 512 x 2048      100  254     0   -1  -1    +1      512  358   -1   +6   -5    +4     1600  631   +2   +9   +1    -7
//   32, 4, 1024 x 2048     128  255    -2   -3  -4    +1      512  345   +3   +7   -1    -2     1600  604   +5   +9   +4   -14
//   64, 8, 1024 x 4096     100  522   -26  -10 -10    -2      512  692  +12  +32   +8    +1     1600 1304  +13  +48  +10   -14
//   128, 8, 768 x 4096     100  550    -3   +1  -1     0      512  778   -8  +11   +1   +29     1600 1383   +2  +42   +3    +8
//   8, 2, 7168 x 4096      100  530    +7   +2  -2    -2      512  685  +70  +33  +11    +8     1600 1403 +178  +61  +18   +28
//   16, 2, 2048 x 8192     100  676    +4   +6  +3    -1      512 1021  +16  +37   +7    +6     1600 2271  +41  +43  +27   -63
// An expert after the other reads weights as one run, which counts while there is little else to do; experts that are chosen unevenly then make
// unequal runs for the XCDs.  Tiles of 160 tokens gain where more than 128 choose most experts and fewer than 160, which the mean does
// not tell: 1.2 % slower in the mean of these and 280 more.
inline ExpertPlan expert_plan(uint32_t n, const ExpertShape &e)
{
    constexpr double kEnds = 10;
    const double mean = (double)n * e.top / e.experts, tiles = e.experts * expert_tiles(mean, kBfTile), share = std::fmin(1.0, (double)n * e.top / (tiles * kBfTile) + 0.125);
    auto kind = [&](uint32_t rows, uint32_t kp) {
        const double steps = kp / kBfStep, wide = bf_wide_step(kBfOffers[0], (rows + 255) / 256 * tiles) * bf_part(share) * steps + kEnds;
        return bf_small_step((rows + 127) / 128 * tiles) * steps < wide ? BfTiles::k128 : BfTiles::kWide;
    };
    return {kind(e.rows, e.kp), kind(e.down_rows, e.down_kp), e.experts >= 128 || (e.experts >= 64 && mean < 32)};
}

}  // namespace lv
