// lv_mid.h — products of steps of 17 to 256 tokens of LLaMA models: the short copy's weights (lv_short.h), activations as two fp16
// halves through LDS.  Up to 64 tokens the smaller ones stay with lv_short.h (short_pays).
//
// Every weight is read once per 128 tokens and unpacked once, for all of a workgroup's tokens; a workgroup of eight waves owns
// RT = RG RTW tiles of 16 rows, T tiles of 16 tokens and all of K or a slice of it.  RG groups of waves take RTW row tiles each, their
// KG = 8 / RG waves deal the K range among themselves, a chunk of four quant blocks at a time, and add up through LDS at the end.
// What bounds such a product besides its bytes and its matrix instructions is the activations' way from L2: 64 bytes a clock into a
// CU, four bytes a token and column, for every workgroup.  Hence many row tiles a workgroup, one copy of the activations in LDS for
// all of them, written by direct loads (no registers), two or three stages ahead of the products: a stage is a block of every K group for
// all T token tiles or half of them.  Weights go from memory to registers, a chunk ahead.
//
// Measured, us, 7B q8_0, gate and up: 48 tokens 47 -> 32 (three row tiles a workgroup, activations through registers, before), 128 tokens
// 92 -> 54 (tiles of 256 rows x 128 tokens on the prompt copy, 88 workgroups); q, k and v 26 -> 22, 89 -> 39.  At 48 tokens the loads alone
// take 28 (the weights alone 22, the activations alone 15), the arithmetic alone 20, launch and sum 7 of each: loads bound it, the activations'
// beside the weights' (vector units at work 42 % of the time, matrix cores 27).  The barrier in the
// middle of a stage and everything read a token tile ahead instead of at its start: 128 tokens 60 -> 54.
#pragma once

#include "lv_short.h"

namespace lv {

constexpr uint32_t kMidTokens = 256;

struct MidArgs {
    // halves of x: element k of token t at x[half] + k / 32 xb + t / 128 x128 + t % 128 / 16 xt + k % 32 / 8 xg + t % 16 16 + k % 8 2
    const uint8_t *x[2];
    uint32_t xb, xt, xg, x128, x_bytes;
    const uint8_t *w;          // short copy of the matrices: kShortQkv: q, k, v one behind the other; kShortSilu: W3 and W1 in pairs
    uint32_t tiles_m, tiles;   // row tiles of a matrix, of the launch
    uint32_t nb;               // blocks of a row, a multiple of 4
    uint32_t slice_chunks;     // chunks of four blocks per K slice (blockIdx.y)
    uint32_t n, mode;
    float *out[kShortSlices];  // [n][ldo], one per slice; kShortQkv: out[0] = q
    uint32_t ldo;
    const float *xscale;       // null, or per token the power of two its halves have to be multiplied by
    uint16_t *cache[2];        // kShortQkv: k and v rows
    const uint32_t *pos_ptr;
    uint32_t pos_add, backlog;
    uint8_t *ff[2];            // kShortSilu: halves of the next product's activations, addressed as x is
    uint32_t fb, ft, fg, f128;
};

// token tiles of a stage: all, or half of what would leave room for two stages only
constexpr int mid_stage_tiles(int t, int rg) { return t > (rg == 1 ? 3 : 5) ? t / 2 : t; }
constexpr int mid_stage_bytes(int t, int rg) { return 8 / rg * 2 * mid_stage_tiles(t, rg) * 1024; }
constexpr int mid_stages(int t, int rg) { return 144 * 1024 / mid_stage_bytes(t, rg) < 4 ? 144 * 1024 / mid_stage_bytes(t, rg) : 4; }
// token tiles whose sums are put together at a time
constexpr int mid_round(int t, int rg, int rtw)
{
    int r = t;
    while (r * rg * rtw * (8 / rg) > 128) r = (r + 1) / 2;
    return r;
}
constexpr int mid_lds_bytes(int t, int rg, int rtw)
{
    const int pipe = mid_stages(t, rg) * mid_stage_bytes(t, rg), sums = mid_round(t, rg, rtw) * rg * rtw * (8 / rg) * 1024;
    return pipe > sums ? pipe : sums;
}

// 16 bytes a lane from base + lane_at + at to 1 KB of LDS.  A buffer load: the compiler takes a global one into LDS for a flat access, behind
// which it waits for all loads at once.
__device__ __forceinline__ void mid_load_lds(const uint8_t *base, uint32_t bytes, uint8_t *lds, int lane_at, uint32_t at)
{
    __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(base), 0, bytes, 0x00020000), (lv_lds_void *)lds, 16, lane_at, at, 0, 0);
}

template <int QT, bool SF32, int T, int RG, int RTW>
__global__ __launch_bounds__(512) void wide_short_gemm_kernel(MidArgs a)
{
    constexpr int KG = 8 / RG, RT = RG * RTW, TS = mid_stage_tiles(T, RG), H = T / TS, NOP = 2 * TS, LPW = NOP / RG;
    constexpr int STAGE = mid_stage_bytes(T, RG), NST = mid_stages(T, RG), TR = mid_round(T, RG, RTW);
    constexpr int CW = QT == 4 ? 4 : 8, CB = short_chunk_bytes(QT, SF32), WL = RTW * (CW / 4 + 1);
    static_assert(NST >= 3 && NOP % RG == 0 && TS * H == T && TS >= 2, "stages");
    extern __shared__ __attribute__((aligned(1024))) uint8_t mid_lds[];
    const int lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rg = wave % RG, kg = wave / RG;
    const uint32_t tile0 = blockIdx.x * RT, tok_tile0 = blockIdx.z * T;
    const uint32_t c0 = blockIdx.y * a.slice_chunks, chunks = min(a.slice_chunks, a.nb / 4 - c0), steps = (chunks + KG - 1) / KG;

    // direct loads of this wave: operand RG p + rg of its K group's block, p = 0 .. LPW - 1 (two row groups: a half each)
    const int x_lane = g * a.xg + r16 * 16;
    uint32_t xo[H][LPW];
#pragma unroll
    for (int h = 0; h < H; h++)
#pragma unroll
        for (int p = 0; p < LPW; p++) {
            const uint32_t t = tok_tile0 + h * TS + (p * RG + rg) / 2;
            xo[h][p] = (t >> 3) * a.x128 + (t & 7) * a.xt;
        }
    // Stage v = (4 j + s) H + h: block s of every K group's chunk j, part h of the token tiles.  Past the end the last block again into a free
    // stage, so that the number of loads in flight stays the same.
    auto issue = [&](uint32_t v, int h, uint32_t slot) {
        const uint32_t u = v / H, c = min(kg + KG * (u >> 2), chunks - 1);
        const uint32_t at = ((c0 + c) * 4 + (u & 3)) * a.xb;
#pragma unroll
        for (int p = 0; p < LPW; p++)
            mid_load_lds(a.x[RG == 2 ? rg : p & 1], a.x_bytes, mid_lds + slot * STAGE + (kg * NOP + p * RG + rg) * 1024, x_lane, xo[h][p] + at);
    };
    // uniform bases of the row tiles (past the last one: the last one again, not stored)
    const uint8_t *wb[RTW];
#pragma unroll
    for (int i = 0; i < RTW; i++) wb[i] = a.w + (size_t)min(tile0 + rg * RTW + i, a.tiles - 1) * short_tile_bytes(QT, SF32, a.nb) + (size_t)(c0 + kg) * CB;
    uint32_t cq[RTW][CW];
    std::conditional_t<SF32, lv_u4, lv_u2> sq[RTW];
    auto fetch_w = [&](uint32_t j) {                   // past the end: one address for all lanes
        const bool ok = kg + KG * j < chunks;
        const uint32_t at = ok ? j * (KG * CB) : 0, lw = ok ? lane * 16 : 0, ls = ok ? r16 * (SF32 ? 16 : 8) : 0;
        const size_t back = ok || kg < (int)chunks ? 0 : (size_t)kg * CB;      // a group without any chunk: the slice's first
#pragma unroll
        for (int i = 0; i < RTW; i++) {
            const uint8_t *p = wb[i] - back;
#pragma unroll
            for (int q = 0; q < CW / 4; q++) {
                const lv_u4 v = *reinterpret_cast<const lv_u4 *>(p + (lw + at + q * 1024));
                cq[i][4 * q] = v.x; cq[i][4 * q + 1] = v.y; cq[i][4 * q + 2] = v.z; cq[i][4 * q + 3] = v.w;
            }
            sq[i] = *reinterpret_cast<const decltype(sq[0] + sq[0]) *>(p + (ls + at + CW / 4 * 1024));
        }
    };

    lv_f4v acc[RTW][T];
#pragma unroll
    for (int i = 0; i < RTW; i++)
#pragma unroll
        for (int t = 0; t < T; t++) acc[i][t] = lv_f4v{0.f, 0.f, 0.f, 0.f};
    const lv_f4v zero = {0.f, 0.f, 0.f, 0.f};

    auto unpack = [&](const uint32_t (&w)[RTW][CW], int i, int s) {
        return QT == 4 ? short_unpack4(w[i][s]) : short_unpack8(w[i][CW / 4 * s], w[i][CW / 4 * s + CW / 8]);
    };

    fetch_w(0);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int v = 0; v < NST - 1; v++) issue(v, v % H, v);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 2) * LPW) : "memory");
    if constexpr (RG > 1) __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    // What a token tile's products need is read or unpacked during the tile before, also from one stage to the next; its sums are scaled and
    // added during the tile behind.
    lv_h8 xh[2], xl[2], b[RTW], bn[RTW];
    auto read_x = [&](int into, uint32_t slot, int t) {
        const uint8_t *xs = mid_lds + slot * STAGE + kg * NOP * 1024 + lane * 16;
        xh[into] = *reinterpret_cast<const lv_h8 *>(xs + 2 * t * 1024);
        xl[into] = *reinterpret_cast<const lv_h8 *>(xs + (2 * t + 1) * 1024);
    };
    read_x(0, 0, 0);
#pragma unroll
    for (int i = 0; i < RTW; i++) b[i] = unpack(cq, i, 0);
    uint32_t slot = 0;
    for (uint32_t j = 0; j < steps; j++) {
        uint32_t w[RTW][CW];
        float sc[RTW][4];
        const bool live = kg + KG * j < chunks;        // not: what the loads past the end returned counts nothing
#pragma unroll
        for (int i = 0; i < RTW; i++) {
#pragma unroll
            for (int q = 0; q < CW; q++) w[i][q] = cq[i][q];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                float d;
                if constexpr (SF32) d = __uint_as_float(sq[i][q]);
                else d = half_bits_to_float((uint16_t)(sq[i][q / 2] >> (16 * (q & 1))));
                sc[i][q] = live ? d : 0.f;
            }
        }
        lv_f4v p[2][RTW];
#pragma unroll
        for (int v = 0; v < 4 * H; v++) {              // stage 4 H j + v
            const int s = v / H, h = v % H;
            const uint32_t next = slot + 1 == NST ? 0 : slot + 1;
#pragma unroll
            for (int t = 0; t < TS; t++) {
                const int n = v * TS + t;              // tiles since the chunk began
                if (t + 1 < TS) read_x((n + 1) & 1, slot, t + 1);
                else read_x((n + 1) & 1, next, 0);
#pragma unroll
                for (int i = 0; i < RTW; i++) p[n & 1][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl[n & 1], b[i], zero, 0, 0, 0);
                if (n > 0) {                           // the tile before
                    const int pt = t > 0 ? h * TS + t - 1 : (h > 0 ? h : H) * TS - 1, ps = t > 0 || h > 0 ? s : s - 1;
#pragma unroll
                    for (int i = 0; i < RTW; i++)
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[i][pt][e] = fmaf(p[(n - 1) & 1][i][e], sc[i][ps], acc[i][pt][e]);
                }
                if (h == H - 1) {                      // the next block's weights, dealt over the tiles
#pragma unroll
                    for (int i = t * RTW / TS; i < (t + 1) * RTW / TS; i++) bn[i] = s < 3 ? unpack(w, i, s + 1) : unpack(cq, i, 0);
                }
#pragma unroll
                for (int i = 0; i < RTW; i++) p[n & 1][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[n & 1], b[i], p[n & 1][i], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (t == 0) {
                    // This wave's loads of the next stage have landed once at most those behind them are in flight: the stages after it and, if
                    // a chunk of weights was asked for since, those.  Behind the barrier its K group's other loads have landed as well, and
                    // everyone is done with the stage before this one, whose place the next loads take.
                    const bool weights_since = v == 1 || (NST == 4 && v == 2);
                    if (weights_since) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 3) * LPW + WL) : "memory");
                    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 3) * LPW) : "memory");
                    if constexpr (RG > 1) __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                    issue(4 * H * j + v + NST - 1, (v + NST - 1) % H, slot == 0 ? NST - 1 : slot - 1);
                    asm volatile("" ::: "memory");
                    if (v == 0) {
                        fetch_w(j + 1);
                        asm volatile("" ::: "memory");
                    }
                }
            }
            if (h == H - 1) {
#pragma unroll
                for (int i = 0; i < RTW; i++) b[i] = bn[i];
            }
            slot = next;
        }
        constexpr int last = 4 * T - 1;
#pragma unroll
        for (int i = 0; i < RTW; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) acc[i][T - 1][e] = fmaf(p[last & 1][i][e], sc[i][3], acc[i][T - 1][e]);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the repeats have landed before the sums take their place

    // ---- the K groups' sums, TR token tiles at a time, through LDS: [row tile][token tile][K group][lane] float4 ------------------
    // acc[i][t][e]: row r16 of row tile i, token 16 t + 4 g + e
    const uint32_t row_at = (a.mode == kShortQkv && a.pos_ptr ? *a.pos_ptr : 0u) + a.pos_add;
    float *const out = a.out[blockIdx.y];
    lv_f4v *const red = reinterpret_cast<lv_f4v *>(mid_lds);
#pragma unroll
    for (int t0 = 0; t0 < T; t0 += TR) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < RTW; i++)
#pragma unroll
            for (int t = 0; t < TR; t++)
                if (t0 + t < T) red[(((rg * RTW + i) * TR + t) * KG + kg) * 64 + lane] = acc[i][t0 + t];
        __syncthreads();
        for (int u = wave; u < RT * TR; u += 8) {
            const uint32_t tile = tile0 + u / TR, tt = t0 + u % TR, tok0 = (tok_tile0 + tt) * 16 + 4 * g;
            if (tile >= a.tiles || tt >= T || (tok_tile0 + tt) * 16 >= a.n) continue;
            float4 xs = make_float4(1.f, 1.f, 1.f, 1.f);
            if (a.xscale) xs = *reinterpret_cast<const float4 *>(a.xscale + tok0);
            auto total = [&](int from, float (&v)[4]) {
                const lv_f4v *src = red + (size_t)u * KG * 64 + from;
                lv_f4v s = src[0];
#pragma unroll
                for (int k = 1; k < KG; k++) s += src[k * 64];
                v[0] = s[0] * xs.x; v[1] = s[1] * xs.y; v[2] = s[2] * xs.z; v[3] = s[3] * xs.w;
            };
            float v[4];
            total(lane, v);
            if (a.mode == kShortSilu) {                // rows 0 .. 7 of the tile are W3's, 8 .. 15 the same ones of W1
                if (r16 >= 8) continue;
                float w1[4];
                total(lane + 8, w1);
                const uint32_t f = tile * 8 + r16;
                const size_t at = (size_t)(f / 32) * a.fb + (size_t)(tok0 / 128) * a.f128 + tok0 % 128 / 16 * a.ft + f % 32 / 8 * a.fg + tok0 % 16 * 16 + f % 8 * 2;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if (tok0 + e >= a.n) continue;
                    const float y = v[e] * w1[e] / (__expf(-w1[e]) + 1.f);
                    const uint16_t h = float_to_half_bits(y);
                    *reinterpret_cast<uint16_t *>(a.ff[0] + at + e * 16) = h;
                    *reinterpret_cast<uint16_t *>(a.ff[1] + at + e * 16) = float_to_half_bits(y - half_bits_to_float(h));
                }
                continue;
            }
            const uint32_t z = tile / a.tiles_m, m = tile % a.tiles_m * 16 + r16;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t tok = tok0 + e;
                if (tok >= a.n) continue;
                if (z == 0) out[(size_t)tok * a.ldo + m] = v[e];
                else if (row_at + tok < a.backlog) a.cache[z - 1][(size_t)(row_at + tok) * a.ldo + m] = float_to_half_bits(v[e]);
            }
        }
    }
}

}  // namespace lv
