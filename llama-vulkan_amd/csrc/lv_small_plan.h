// lv_small_plan.h — which models take lv_small.h's launch for a token, with how many workgroups, and up to which context.
#pragma once

#include <algorithm>
#include <cstdint>

namespace lv {

constexpr int kSmallThreads = 512, kSmallWaves = kSmallThreads / 64;
constexpr uint32_t kSmallMaxDim = 1024;    // two values of a normalised vector a thread
constexpr uint32_t kSmallMaxFf = 8192;     // floats of LDS
constexpr uint32_t kSmallMaxWGs = 64;      // each waits for the others: all of them, of four launches at once, find room beside one another
constexpr uint32_t kSmallPartBlocks = 4;   // blocks a thread multiplies of a workgroup's own columns of Wo or W2, at most

// lanes a row of nb blocks, as a power of two
constexpr int small_lanes_log2(uint32_t nb) { return nb <= 8 ? 3 : nb <= 16 ? 4 : nb <= 32 ? 5 : 6; }
// o, x1, ff, x2; with partial sums: one vector of every head and of every workgroup that has feed-forward blocks
constexpr uint32_t small_parts(uint32_t F, uint32_t own) { return (F / 32 + own - 1) / own; }
constexpr uint32_t small_layer_floats(uint32_t D, uint32_t F, uint32_t heads, uint32_t own) { return own ? (heads + small_parts(F, own)) * D : 3 * D + F; }

// Which models take lv_small.h's launch for a token: those whose operator chain has ten launches a layer (below the streaming kernels' 2048
// rows) and whose work a few workgroups do in less time than those launches take to follow one another.  A head's three projections are one
// workgroup's work, at most kSmallHeadTiles tiles a wave were looked at; then both times are estimated, in us behind 100 rows of context:
//   launch  17 + layers (9.6 + 1.1 tiles a wave of a head's projections + 0.95 tiles a wave of the other products) + 1.26 of the output's
//           + 0.1 for 1000 logits; partial sums (below) 1.5 less a layer
//   chain   25 + layers (42 + 0.125 MB) + 0.06 MB of the output + 0.27 for 1000 logits, which it copies
// a fit of shapes of width 64 to 1024, 300 to 128256 rows of output, steps whose logits are read; over 140 of them 13 % off either way's
// measured times at most (partial sums 16 %).
// Measured, launch and chain: width 256, 2 layers 47 and 117; 512, 8 layers 198 and 361; 768, 12 layers 464 and 568.  A large vocabulary is
// what a quarter of the chip is too little for: 640 wide, 4 layers, 128256 rows 260 and 240, 1024, 1 layer, 203 and 116; of a narrow
// model it is not: 256, 1 layer, 128256 rows 87 and 106, 128 wide 91 and 107.
constexpr uint32_t kSmallHeadTiles = 12;
// One workgroup also walks a head's cache rows, where the chain splits them over several: 80 ns more of a layer for every 1000 elements of
// them, so what the launch gains bounds the context, and so do the rows that were looked at.  Width 512, 4 heads of 128, 4 layers 148 and
// 191 us behind 100 rows, 199 and 205 behind 1000, 257 and 221 behind 2000; width 256, 4 heads of 64, 76 and 118 behind 2000.
constexpr uint32_t kSmallRowElements = 131072;
// Partial sums (lv_small.h) save two hand-overs a layer, 4 to 5 us, and every workgroup reads (heads + parts) D floats a layer instead of
// 3 D + F and unpacks blocks row by row.  us a token, 4 layers unless said, without and with them, q4_0 and q8_0: width 128 and 352 84 74, 86 82;
// 256 and 704 88 75, 89 78, 8 layers and 32000 rows of output 156 146, 159 153; 256 and 4096 (two blocks a workgroup) 85 79, 87 83;
// 288 and 768 87 82, 88 85, 32000 rows 112 107, 112 111, and there behind 600 rows 118 117, 120 120.  Above, what is gained with a short context
// and few rows of output is lost otherwise: 320 and 1280, 10 heads 88 83, 89 86, with 32000 rows behind 600 120 120, 122 124; 384 and 1024
// 161 165, 162 170; 448 and 1216 102 98, 104 104, with 32000 rows 124 127, 126 131; 512 and 1376 98 96, 100 102; 576 and 1536 134 141.
constexpr uint32_t kSmallPartDim = 288;

struct SmallShape {
    uint32_t D, F, heads, rot, layers, vocab, block_bytes;      // block_bytes: of 32 weights, 18 or 34
};
struct SmallPlan {
    uint32_t wgs = 0;           // workgroups of the launch, 0: the chain
    uint32_t own = 0;           // with partial sums: feed-forward blocks of a workgroup, a power of two; 0: four hand-overs a layer
    uint32_t elements = 0;      // cache elements of a head up to which it is the faster way
};
inline SmallPlan small_plan(const SmallShape &m)
{
    if (m.D > kSmallMaxDim || m.F > kSmallMaxFf || m.heads > kSmallMaxWGs) return {};
    // tiles of `waves` waves of a matrix, the longest wave's
    const auto tiles = [](uint32_t rows, uint32_t cols, uint32_t waves) -> uint32_t {
        const uint32_t nb = cols / 32, lanes = 1u << small_lanes_log2(nb);
        return ((rows * lanes + 63) / 64 + waves - 1) / waves * ((nb + lanes - 1) / lanes);
    };
    const uint32_t head = tiles(3 * m.rot, m.D, kSmallWaves);
    if (head > kSmallHeadTiles) return {};
    // a pair of tiles a wave in the feed-forward, or four tiles of a large vocabulary
    const uint32_t most = std::max(tiles(m.F, m.D, 1), tiles(m.vocab, m.D, 1) / 4);
    SmallPlan p;
    p.wgs = std::min(kSmallMaxWGs, std::max(m.heads, (most + kSmallWaves - 1) / kSmallWaves));
    if (m.D <= kSmallPartDim) {
        const uint32_t own = small_parts(m.F, 1) <= kSmallMaxWGs ? 1 : 2, parts = small_parts(m.F, own);
        if (parts <= kSmallMaxWGs && m.D * std::max(own, m.rot / 32) <= kSmallPartBlocks * kSmallThreads) {
            p.own = own;
            p.wgs = std::max(p.wgs, parts);
        }
    }
    const uint32_t waves = p.wgs * kSmallWaves;
    const double mb = m.block_bytes / 32e6, layer_mb = (4.0 * m.D * m.D + 3.0 * m.D * m.F) * mb, output_mb = (double)m.vocab * m.D * mb;
    const double products = 0.95 * (tiles(m.D, m.D, waves) + 2 * tiles(m.F, m.D, waves) + tiles(m.D, m.F, waves));
    const double launch = 17 + m.layers * (9.6 + 1.1 * head + products - (p.own ? 1.5 : 0.0)) + 1.26 * tiles(m.vocab, m.D, waves) + 0.1e-3 * m.vocab;
    const double chain = 25 + m.layers * (42 + 0.125 * layer_mb) + 0.06 * output_mb + 0.27e-3 * m.vocab;
    if (launch >= chain) return {};
    p.elements = (uint32_t)std::min<double>(kSmallRowElements, (chain - launch) / m.layers / 0.08 * 1000);
    return p;
}

}  // namespace lv
