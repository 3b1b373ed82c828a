// lv_short.h — short batches (2 .. 64 tokens: a command, the next message of a chat) of LLaMA models: products with the
// quantised matrices as the operator path stores them, and attention split over cache positions.
//
// What bounds such a step is reading the weights once.  The GEMM of lv_gemm.h reads a copy of 2.1 bytes a weight and works on tiles
// of 128 tokens; the persistent kernel reads all weights per token.  Here every weight is read once, in its 4.5 or 8.5 bits, and
// unpacked in registers on its way into the matrix cores.  Every product is exact, a block's 32 products are summed in fp32, then
// multiplied by the block's scale and added to the fp32 result.  Activations:
//   up to 16 tokens   three bf16 parts, an exact cut of the fp32 value with all of its range.  Such a step is also evaluated token by
//                     token (other paths, no room for the copy below), in fp32 throughout, and is held to the same.
//   17 to 64          two fp16 halves as in lv_gemm.h, which takes longer steps and these without the copy: 22 bits, of the norms'
//                     outputs scaled per token; feed-forward and attention outputs unscaled, below 65504.  Their products: lv_mid.h,
//                     smaller ones here.
// Attention likewise: up to 15 tokens in fp32 (short_attn_exact_kernel), then short_attn_kernel on fp16 pairs as with longer steps.
//
// short_gemm_kernel.  A workgroup of 8 waves owns RT tiles of 16 weight rows over all of K (or one of up to 4 slices of it) and all
// tokens; its waves deal the K range among themselves, four quant blocks at a time, and add up through LDS at the end.  A wave so
// reads activations nobody else in the workgroup reads, straight into MFMA operand form, and reuses them for its RT tiles: no
// LDS, no barrier, nothing but loads in flight in the main loop.
//   weights ("short copy", made when a model evaluates its first short batch; as many bytes as the file has):
//       [row tile of 16][chunk of 4 blocks][64 lanes][dwords of blocks 0 .. 3][16 rows][4 scales, fp16 or (version-1 files) fp32]
//       A lane's codes of a block are the eight it feeds to one MFMA (v_mfma_f32_16x16x32_f16: lane l holds row l % 16, k group l / 16), so
//       a load is 1 KB in a row and nothing crosses lanes.  Read from the operator path's planes instead, a load touches 16 rows,
//       16 consecutive lanes 16 cache lines: the address path, not HBM, then sets the time (7B q4_0 gate and up for 8 tokens: 21.5 us that way, 15.8 so).
//   order: the eight codes a lane feeds to an MFMA come in the order that unpacks cheapest (short_slot); activation parts are
//          written in that order, the nibbles of q4_0 packed so that halves stay in order.
//   activations: [block][16-token tile][operand][group][token][8 elements]: 1 KB per operand, a lane's 16 bytes at 16 l.  Up to 8 tokens:
//          the first two parts share an operand (tokens 0 .. 7 and 8 .. 15 of it), the third is half of one.
// Rows of tokens past the batch are not written; a token only meets its own row of the result.
//
// Norms of up to 16 tokens have no launch of their own: the norm is (x w) / rms with one number a token.  The last of a row group's K
// slices to arrive (kShortResidual) adds them to x, writes the parts of x w and the group's sum and squared deviations of x; the next
// product puts those together while its first weights are on their way, and multiplies its results by 1 / rms.  A norm's launch is one
// workgroup a token, 5.6 us of latency on eight CUs; putting slices together takes 2.9 at the end of the product (7B q4_0, 8 tokens: a
// layer's two products and norms 26.8 -> 21.4 us, the step 2.00 -> 1.82 ms).  Halves need the row's largest value before they are made
// and keep short_norm_kernel.
//
// Measured (us per launch, 7B layer, 8 tokens q4_0): q, k and v 11, gate and up 16, attention output 9 and down 12.5; about 3 of each
// launch and sum.  While they run the vector units are at work 48 % of the time in gate and up, 42 in q, k and v, 30 in the others, the matrix
// cores 22, 19 and 15, and a wave waits to issue a fifth to a third of its own: no one unit bounds them.  A step of 8 tokens, 7B q4_0:
// 7.31 -> 1.82 ms (eight launches of the persistent kernel before).
#pragma once

#include "lv_attn_batch.h"
#include "lv_gemm.h"
#include "lv_mega.h"

namespace lv {

constexpr uint32_t kShortTokens = 64;
constexpr uint32_t kShortExact = 16;       // tokens of steps on three parts
constexpr uint32_t kShortStatLanes = 4;    // row groups a lane of a wave adds up: 256 of at least 32 rows, up to 8192
constexpr int kShortWaves = 8;
constexpr int kShortSlices = kGemmMaxMats;

typedef _Float16 lv_h2 __attribute__((ext_vector_type(2)));
typedef uint32_t lv_u4 __attribute__((ext_vector_type(4)));
typedef __bf16 lv_b2 __attribute__((ext_vector_type(2)));
typedef uint32_t lv_u2 __attribute__((ext_vector_type(2)));

// tiles of 16 tokens; 0: up to 8 tokens, whose parts share operands
__host__ __device__ constexpr uint32_t short_tiles(uint32_t n) { return n <= 8 ? 0 : (n + 15) / 16; }
// three bf16 parts, not two fp16 halves: up to 16 tokens
__host__ __device__ constexpr bool short_exact(uint32_t tiles) { return tiles <= kShortExact / 16; }
__host__ __device__ constexpr uint32_t short_block_bytes(uint32_t tiles) { return tiles == 0 ? 1536 : tiles == 1 ? 3072 : tiles * 2048; }
// bytes of the activations of K columns
__host__ __device__ constexpr size_t short_act_bytes(uint32_t K, uint32_t n) { return (size_t)(K / 32) * short_block_bytes(short_tiles(n)); }

// Element k of a block (0 .. 31) -> slot 8 g + e of the operand: group g holds elements 8g .. 8g + 7.  Halves and q8_0: in order.  Parts of
// q4_0: nibble p of a lane's dword holds element 2 (p % 4) + p / 4 (a masked dword leaves nibbles 0 and 4, then 1 and 5, 2 and 6, 3 and 7 in
// the two halves of a register, in order), and the conversion from bytes takes the low nibbles first, then the high ones: 0 4 1 5 2 6 3 7.
template <int QT, bool PARTS>
__host__ __device__ constexpr uint32_t short_slot(uint32_t k)
{
    if constexpr (QT == 8 || !PARTS) return k;
    return (k & ~7u) + (k & 3) * 2 + ((k >> 2) & 1);
}
// the elements of a group, slots 0 .. 7, from its two runs of four consecutive elements
template <int QT>
__device__ __forceinline__ void short_order(float (&f)[8], const float4 &a, const float4 &b, bool parts)
{
    if (QT == 8 || !parts) {
        f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w; f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
    } else {
        f[0] = a.x; f[1] = b.x; f[2] = a.y; f[3] = b.y; f[4] = a.z; f[5] = b.z; f[6] = a.w; f[7] = b.w;
    }
}

// where part `part` of (block, token, group) lies: 0, 1 and 2, or the halves 0 and 1
__device__ __forceinline__ size_t short_act_offset(uint32_t block, uint32_t token, uint32_t g, uint32_t tiles, uint32_t part)
{
    const size_t at = (size_t)block * short_block_bytes(tiles);
    if (tiles == 0) return at + (part < 2 ? g * 256 + part * 128 : 1024 + g * 128) + token * 16;
    return at + token / 16 * 2048 + part * 1024 + (g * 16 + token % 16) * 16;
}
// x = b[0] + b[1] + b[2], each the upper half of its dword: eight bits a part
__device__ __forceinline__ void short_cut(uint32_t (&b)[3], float x)
{
    b[0] = __float_as_uint(x) & 0xffff0000u;
    const float r = x - __uint_as_float(b[0]);
    b[1] = __float_as_uint(r) & 0xffff0000u;
    b[2] = __float_as_uint(r - __uint_as_float(b[1]));
}
// the eight elements of (block, token, group)
__device__ __forceinline__ void short_put(uint8_t *act, uint32_t block, uint32_t token, uint32_t g, uint32_t tiles, const float (&f)[8])
{
    uint4 p[3];
    if (short_exact(tiles)) {
        uint32_t w[3][4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            uint32_t b0[3], b1[3];
            short_cut(b0, f[2 * j]);
            short_cut(b1, f[2 * j + 1]);
#pragma unroll
            for (int i = 0; i < 3; i++) w[i][j] = (b0[i] >> 16) | (b1[i] & 0xffff0000u);
        }
#pragma unroll
        for (int i = 0; i < 3; i++) p[i] = make_uint4(w[i][0], w[i][1], w[i][2], w[i][3]);
        *reinterpret_cast<uint4 *>(act + short_act_offset(block, token, g, tiles, 2)) = p[2];
    } else {
        gemm_split8(p[0], p[1], f);
    }
    *reinterpret_cast<uint4 *>(act + short_act_offset(block, token, g, tiles, 0)) = p[0];
    *reinterpret_cast<uint4 *>(act + short_act_offset(block, token, g, tiles, 1)) = p[1];
}

enum ShortMode { kShortStore = 0, kShortQkv = 1, kShortSilu = 2, kShortResidual = 3 };

struct ShortArgs {
    const uint8_t *x;          // activations
    const uint8_t *w;          // short copy of the matrices: kShortQkv: q, k, v one behind the other; kShortSilu: W3 and W1 in pairs
    uint32_t tiles_m, tiles;   // row tiles of a matrix, of the launch
    uint32_t nb;               // blocks of a row, a multiple of 4
    uint32_t slice_chunks;     // chunks of four blocks per K slice (blockIdx.y)
    uint32_t n, mode;
    float *out[kShortSlices];  // [n][ldo], one per slice; kShortQkv: out[0] = q
    uint32_t ldo;
    const float *xscale;       // null, or per token the power of two its halves have to be multiplied by (not with parts)
    uint16_t *cache[2];        // kShortQkv: k and v rows
    const uint32_t *pos_ptr;
    uint32_t pos_add, backlog;
    uint8_t *ff;               // kShortSilu: activations of the next product
    // kShortResidual, up to 16 tokens: x += the product, x w as the next product's activations, and sum and squared deviations of x by row
    // groups (a workgroup's rows) and tokens.  The last of a row group's K slices to arrive does it; counters are zero before and after.
    float *res;                // x, [n][ldo]
    const float *norm_w;
    uint8_t *act_out;
    float2 *stats_out;         // [row group][kShortExact]
    uint32_t *counters;        // [row group]
    // Input of parts of x w: the results are multiplied by the tokens' 1 / rms, from these of `stat_groups` groups of `stat_rows` rows
    const float2 *stats;       // null: the activations are whole
    uint32_t stat_groups, stat_rows, dim;
};

// Loads of a chunk are requested while the one before it is multiplied, activations as far ahead as the weights or, where a block's
// products take long enough to cover an L2 access, two blocks ahead.  More in flight per wave costs registers, hence waves per
// CU, and lost (two chunks of weights: 7B q4_0 gate and up for 8 tokens 15.8 -> 16.5 us).  Nor do two workgroups a CU pay: two blocks
// ahead would let three row tiles of q4_0 and up to 16 tokens into 128 registers (a step of 8 tokens of 13B q4_0, 8 layers: 752 us so,
// 708 with four ahead).
template <int T, int RT> constexpr int short_ahead() { return T * RT >= 8 ? 2 : 4; }
// RT tiles of rows beside T tiles of tokens that keep sums, queues and activations in 256 registers, and that short_pays asks for
__host__ __device__ constexpr bool short_fits(int qt, uint32_t t, uint32_t rt)
{
    if (t > 2) return rt == 2;
    return rt <= (qt == 8 && t == 2 ? 3u : 6u);
}
// row tiles whose sums are put together at a time: up to 64 KB of LDS, whole pairs
template <int T, int RT> constexpr int short_round()
{
    constexpr int most = 8 / (T ? T : 1);
    return RT <= most ? RT : most;
}
__device__ __forceinline__ lv_h8 short_unpack4(uint32_t w)
{
    // nibble q in the low bits of a half of pattern 0x6400 is 1024 + q; one place up, 1024 + 16 q: both to q - 8, exactly
    const uint32_t v = w >> 8;
    const lv_h2 p0 = __builtin_bit_cast(lv_h2, (w & 0x000f000fu) | 0x64006400u), p1 = __builtin_bit_cast(lv_h2, (w & 0x00f000f0u) | 0x64006400u);
    const lv_h2 p2 = __builtin_bit_cast(lv_h2, (v & 0x000f000fu) | 0x64006400u), p3 = __builtin_bit_cast(lv_h2, (v & 0x00f000f0u) | 0x64006400u);
    const lv_h2 c = {(_Float16)-1032.f, (_Float16)-1032.f}, s = {(_Float16)0.0625f, (_Float16)0.0625f}, d = {(_Float16)-72.f, (_Float16)-72.f};
    union { lv_h2 h[4]; lv_h8 v8; } u;
    u.h[0] = p0 + c;
    u.h[1] = __builtin_elementwise_fma(p1, s, d);
    u.h[2] = p2 + c;
    u.h[3] = __builtin_elementwise_fma(p3, s, d);
    return u.v8;
}
__device__ __forceinline__ lv_h8 short_unpack8(uint32_t lo, uint32_t hi)
{
    // byte b ^ 0x80 under 0x64 is 1024 + 128 + b
    const uint32_t a = lo ^ 0x80808080u, b = hi ^ 0x80808080u;
    const lv_h2 c = {(_Float16)-1152.f, (_Float16)-1152.f};
    union { lv_h2 h[4]; lv_h8 v8; } u;
    u.h[0] = __builtin_bit_cast(lv_h2, __builtin_amdgcn_perm(0x64646464u, a, 0x04010400u)) + c;
    u.h[1] = __builtin_bit_cast(lv_h2, __builtin_amdgcn_perm(0x64646464u, a, 0x04030402u)) + c;
    u.h[2] = __builtin_bit_cast(lv_h2, __builtin_amdgcn_perm(0x64646464u, b, 0x04010400u)) + c;
    u.h[3] = __builtin_bit_cast(lv_h2, __builtin_amdgcn_perm(0x64646464u, b, 0x04030402u)) + c;
    return u.v8;
}
// bf16, q4_0: a byte 0x0q is q 2^-9 as an fp8 number.  The codes stay unsigned: 8 times every activation is taken off the sum instead, as
// with q4_block_dot.
__device__ __forceinline__ lv_b8 short_unpack4_bf16(uint32_t w)
{
    const uint32_t l = w & 0x0f0f0f0fu, h = (w >> 4) & 0x0f0f0f0fu;
    union { lv_b2 h[4]; lv_b8 v8; } u;
    u.h[0] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(l, 512.f, false);
    u.h[1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(l, 512.f, true);
    u.h[2] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(h, 512.f, false);
    u.h[3] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(h, 512.f, true);
    return u.v8;
}
// q8_0: a signed byte converts to fp32, where a whole number of eight bits leaves the lower half zero
__device__ __forceinline__ lv_b8 short_unpack8_bf16(uint32_t lo, uint32_t hi)
{
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t d = (j < 2 ? lo : hi) >> (16 * (j & 1));
        w[j] = __builtin_amdgcn_perm(__float_as_uint((float)(int8_t)(d >> 8)), __float_as_uint((float)(int8_t)d), 0x07060302u);
    }
    return __builtin_bit_cast(lv_b8, lv_u4{w[0], w[1], w[2], w[3]});
}
__host__ __device__ constexpr uint32_t short_chunk_bytes(int qt, bool sf32) { return (qt == 4 ? 1024 : 2048) + (sf32 ? 256 : 128); }
__host__ __device__ constexpr size_t short_tile_bytes(int qt, bool sf32, uint32_t nb) { return (size_t)(nb / 4) * short_chunk_bytes(qt, sf32); }

// The short copy of a matrix, or (PAIR) of W3 and W1 together: tiles of eight rows of W3 and the same eight of W1, so that a workgroup
// has both products of a row whatever its number of tiles.  One thread per (tile, chunk, lane); `tiles` row tiles, nb a multiple of 4.
template <int QT, bool PAIR>
__global__ __launch_bounds__(256) void short_pack_kernel(uint8_t *__restrict__ dst, MatView m, MatView m2, uint32_t tiles)
{
    const uint32_t nb = m.cols / 32, chunks = nb / 4;
    const uint64_t unit = ((uint64_t)blockIdx.x * 256 + threadIdx.x) >> 6;
    const uint32_t lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, c = (uint32_t)(unit % chunks), tile = (uint32_t)(unit / chunks);
    if (tile >= tiles) return;
    const MatView &src = PAIR && r >= 8 ? m2 : m;
    const uint64_t b0 = (uint64_t)(PAIR ? tile * 8 + (r & 7) : tile * 16 + r) * nb + c * 4;
    const bool sf32 = src.scales_f32 != nullptr;
    uint8_t *out = dst + (size_t)tile * short_tile_bytes(QT, sf32, nb) + (size_t)c * short_chunk_bytes(QT, sf32);
    uint32_t w[QT];
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const uint32_t *b = reinterpret_cast<const uint32_t *>(src.codes + (b0 + s) * (QT / 4));
        if constexpr (QT == 4) {
            // elements 8g .. 8g + 7: the low (groups 0 and 1) or high nibbles of eight bytes, to where short_slot wants them
            const uint32_t lo = b[(g & 1) * 2] >> (g >> 1) * 4 & 0x0f0f0f0fu, hi = b[(g & 1) * 2 + 1] >> (g >> 1) * 4 & 0x0f0f0f0fu;
            w[s] = 0;
#pragma unroll
            for (int e = 0; e < 8; e++) w[s] |= ((e < 4 ? lo : hi) >> 8 * (e & 3) & 15u) << 4 * ((e >> 1) + 4 * (e & 1));
        }
        else { w[2 * s] = b[2 * g]; w[2 * s + 1] = b[2 * g + 1]; }
    }
#pragma unroll
    for (int i = 0; i < QT / 4; i++) *reinterpret_cast<uint4 *>(out + i * 1024 + lane * 16) = make_uint4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
    if (g == 0) {
#pragma unroll
        for (int s = 0; s < 4; s++) {
            if (sf32) *reinterpret_cast<float *>(out + QT / 4 * 1024 + r * 16 + s * 4) = src.scales_f32[b0 + s];
            else *reinterpret_cast<uint16_t *>(out + QT / 4 * 1024 + r * 8 + s * 2) = src.scales[b0 + s];
        }
    }
}

// T: tiles of 16 tokens, 0: up to 8 tokens; RT: tiles of 16 rows per workgroup; SF32: fp32 block scales
template <int QT, bool SF32, int T, int RT>
__global__ __launch_bounds__(kShortWaves * 64) void short_gemm_kernel(ShortArgs a)
{
    constexpr bool EIGHT = T == 0;                     // 8 tokens: an operand holds their first parts and their second ones
    constexpr bool EXACT = short_exact(T);
    constexpr int NT = EIGHT ? 1 : T;
    constexpr int XB = short_block_bytes(T);           // activation bytes of a block
    constexpr int NX = EIGHT ? 2 : EXACT ? 3 : 2 * NT; // its operands
    constexpr int BB = QT == 4 ? 16 : 32;              // code bytes of a block
    constexpr int CW = BB / 4;                         // a lane's dwords of a chunk
    constexpr int CB = short_chunk_bytes(QT, SF32);
    constexpr int XD = short_ahead<T, RT>();
    constexpr int PR = short_round<T, RT>();           // row tiles summed at a time
    __shared__ __attribute__((aligned(16))) float red[PR * NT * kShortWaves * 256];
    __shared__ __attribute__((aligned(16))) float inv_rms[EXACT ? kShortExact : 1];
    __shared__ uint32_t arrived;
    const int lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t tile0 = blockIdx.x * RT;
    const uint32_t c0 = blockIdx.y * a.slice_chunks, chunks = min(a.slice_chunks, a.nb / 4 - c0);
    const uint32_t steps = chunks > (uint32_t)wave ? (chunks - wave + kShortWaves - 1) / kShortWaves : 0;
    const uint32_t nb = a.nb;

    // uniform bases of the row tiles (past the last one: the last one again, not stored)
    const uint8_t *wb[RT];
#pragma unroll
    for (int t = 0; t < RT; t++) wb[t] = a.w + (size_t)min(tile0 + t, a.tiles - 1) * short_tile_bytes(QT, SF32, nb) + (size_t)(c0 + wave) * CB;
    const uint8_t *xb = a.x + (size_t)(c0 + wave) * 4 * XB;

    // Loads of chunk j.  They return in the order they were issued, so activations (L2) are requested as far ahead as weights (HBM).
    // Past this wave's last chunk: one address for all lanes, which costs next to nothing and keeps the queue free of branches.
    uint32_t cq[RT][CW];
    std::conditional_t<SF32, lv_u4, lv_u2> sq[RT];
    lv_u4 xq[XD][NX];
    auto fetch_w = [&](uint32_t j) {
        const uint32_t at = j < steps ? j * (kShortWaves * CB) : 0, lw = j < steps ? lane * 16 : 0, ls = j < steps ? r16 * (SF32 ? 16 : 8) : 0;
#pragma unroll
        for (int t = 0; t < RT; t++) {
#pragma unroll
            for (int i = 0; i < CW / 4; i++) {
                const lv_u4 v = *reinterpret_cast<const lv_u4 *>(wb[t] + (lw + at + i * 1024));
                cq[t][4 * i] = v.x; cq[t][4 * i + 1] = v.y; cq[t][4 * i + 2] = v.z; cq[t][4 * i + 3] = v.w;
            }
            sq[t] = *reinterpret_cast<const decltype(sq[0] + sq[0]) *>(wb[t] + (ls + at + CW / 4 * 1024));
        }
    };
    auto fetch_x = [&](int slot, uint32_t j, int s) {  // block s of chunk j
        const uint8_t *p = xb + (j < steps ? ((size_t)j * (kShortWaves * 4) + s) * XB : 0);
        const uint32_t l = j < steps ? lane * 16 : 0;
#pragma unroll
        for (int t = 0; t < NX; t++) {
            const uint32_t at = EIGHT && t == 1 ? (j < steps ? g * 128 + (r16 & 7) * 16 : 0) : l;
            xq[slot][t] = *reinterpret_cast<const lv_u4 *>(p + at + t * 1024);
        }
    };
    lv_f4v acc[RT][NT];
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[i][t] = lv_f4v{0.f, 0.f, 0.f, 0.f};
    const lv_f4v zero = {0.f, 0.f, 0.f, 0.f};
    constexpr uint32_t kOnes = 0x3f803f80u;

    // a wave's tokens: `wave` and, beyond 8, `wave` + 8.  Asked for before the weights, added up while those are on their way.
    constexpr int WT = EIGHT ? 1 : 2;
    float2 st[EXACT ? WT : 1][kShortStatLanes];
    if constexpr (EXACT) {
        if (a.stats) {
#pragma unroll
            for (int t = 0; t < WT; t++)
#pragma unroll
                for (uint32_t j = 0; j < kShortStatLanes; j++) st[t][j] = j * 64 + lane < a.stat_groups ? a.stats[(j * 64 + lane) * kShortExact + wave + 8 * t] : make_float2(0.f, 0.f);
        }
    }
    if (steps) {
        fetch_w(0);
#pragma unroll
        for (int s = 0; s < XD; s++) fetch_x(s, 0, s);
    }
    if constexpr (EXACT) {
        if (a.stats) {
#pragma unroll
            for (int t = 0; t < WT; t++) {
                float sum = 0.f, q = 0.f;
#pragma unroll
                for (uint32_t j = 0; j < kShortStatLanes; j++) sum += st[t][j].x;
                const float mean = wave_sum(sum) / (float)a.dim;
#pragma unroll
                for (uint32_t j = 0; j < kShortStatLanes; j++) {
                    const uint32_t grp = j * 64 + lane;
                    if (grp >= a.stat_groups) continue;
                    const float rows = (float)min(a.stat_rows, a.dim - grp * a.stat_rows), d = st[t][j].x / rows - mean;
                    q += fmaf(rows * d, d, st[t][j].y);
                }
                q = wave_sum(q);
                if (lane == 0) inv_rms[wave + 8 * t] = rsqrtf(q / (float)a.dim);
            }
        }
    }
    if (steps) {
        for (uint32_t j = 0; j < steps; j++) {
            uint32_t w[RT][CW];                        // dword s (q8_0: 2 s and 2 s + 1): this lane's codes of block s
            float sc[RT][4];
#pragma unroll
            for (int t = 0; t < RT; t++) {
#pragma unroll
                for (int i = 0; i < CW; i++) w[t][i] = cq[t][i];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if constexpr (SF32) sc[t][i] = __uint_as_float(sq[t][i]);
                    else sc[t][i] = half_bits_to_float((uint16_t)(sq[t][i / 2] >> (16 * (i & 1))));
                }
            }
            fetch_w(j + 1);
#pragma unroll
            for (int s = 0; s < 4; s++) {
                lv_u4 ax[NX];                          // parts, or high and low halves tile by tile
#pragma unroll
                for (int t = 0; t < NX; t++) ax[t] = xq[s % XD][t];
                if constexpr (EIGHT) ax[1] = r16 >= 8 ? ax[1] : lv_u4{0u, 0u, 0u, 0u};       // the third parts beside the second
                auto times = [&](const lv_b8 &b, lv_f4v c) {       // all parts, the small ones first
#pragma unroll
                    for (int t = NX - 1; t >= 0; t--) c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(lv_b8, ax[t]), b, c, 0, 0, 0);
                    return c;
                };
                lv_f4v from = zero;
                if constexpr (EXACT && QT == 4) from = times(__builtin_bit_cast(lv_b8, lv_u4{kOnes, kOnes, kOnes, kOnes}), zero) * -8.f;
#pragma unroll
                for (int i = 0; i < RT; i++) {
                    lv_f4v p[NT];
                    if constexpr (EXACT) {
                        const lv_b8 b = QT == 4 ? short_unpack4_bf16(w[i][s]) : short_unpack8_bf16(w[i][CW / 4 * s], w[i][CW / 4 * s + CW / 8]);
                        p[0] = times(b, from);
                    } else {
                        const lv_h8 b = QT == 4 ? short_unpack4(w[i][s]) : short_unpack8(w[i][CW / 4 * s], w[i][CW / 4 * s + CW / 8]);
#pragma unroll
                        for (int t = 0; t < NT; t++) p[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(lv_h8, ax[2 * t + 1]), b, zero, 0, 0, 0);
#pragma unroll
                        for (int t = 0; t < NT; t++) p[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(lv_h8, ax[2 * t]), b, p[t], 0, 0, 0);
                    }
#pragma unroll
                    for (int t = 0; t < NT; t++)
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[i][t][e] = fmaf(p[t][e], sc[i][s], acc[i][t][e]);
                }
                fetch_x(s % XD, j + (s + XD) / 4, (s + XD) % 4);
            }
        }
    }

    // ---- the waves' sums, PR row tiles at a time, through LDS: [row tile][token tile][wave][lane] float4 -------------------------
    // acc[i][t][e]: row r16 of row tile i, token 16 t + 4 g + e (EIGHT: the first part's product of token 4 g + e for g < 2, behind
    // them the others').  A wave adds up every eighth (row tile, token tile).
    const uint32_t row_at = (a.mode == kShortQkv && a.pos_ptr ? *a.pos_ptr : 0u) + a.pos_add;
    float *const out = a.out[blockIdx.y];
    auto total = [&](int u, int from, float (&v)[4], const float4 &xs) {      // lane `from`'s sums of unit u
        const lv_f4v *src = reinterpret_cast<const lv_f4v *>(red) + (size_t)u * kShortWaves * 64 + from;
        lv_f4v s = src[0];
#pragma unroll
        for (int w = 1; w < kShortWaves; w++) s += src[w * 64];
        if constexpr (EIGHT) {
            const lv_f4v *low = src + (from < 32 ? 32 : 0);
#pragma unroll
            for (int w = 0; w < kShortWaves; w++) s += low[w * 64];
        }
        v[0] = s[0] * xs.x; v[1] = s[1] * xs.y; v[2] = s[2] * xs.z; v[3] = s[3] * xs.w;
    };
#pragma unroll
    for (int i0 = 0; i0 < RT; i0 += PR) {
        if (i0) __syncthreads();
#pragma unroll
        for (int i = 0; i < PR; i++)
#pragma unroll
            for (int t = 0; t < NT; t++)
                if (i0 + i < RT) *reinterpret_cast<lv_f4v *>(red + (((i * NT + t) * kShortWaves + wave) * 64 + lane) * 4) = acc[i0 + i][t];
        __syncthreads();
        for (int u = wave; u < (RT - i0 < PR ? RT - i0 : PR) * NT; u += kShortWaves) {
            const uint32_t tile = tile0 + i0 + u / NT, tok0 = 16 * (u % NT) + 4 * g;
            if (tile >= a.tiles || (EIGHT && lane >= 32)) continue;
            float4 xs = make_float4(1.f, 1.f, 1.f, 1.f);
            if constexpr (EXACT) {
                if (a.stats) xs = *reinterpret_cast<const float4 *>(inv_rms + tok0);
            } else {
                if (a.xscale) xs = *reinterpret_cast<const float4 *>(a.xscale + tok0);
            }
            float v[4];
            total(u, lane, v, xs);
            if (a.mode == kShortSilu) {                // rows 0 .. 7 of the tile are W3's, 8 .. 15 the same ones of W1
                if (r16 >= 8) continue;
                float w[4];
                total(u, lane + 8, w, xs);
                const uint32_t f = tile * 8 + r16, slot = short_slot<QT, EXACT>(f & 31);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if (tok0 + e >= a.n) continue;
                    const float y = v[e] * w[e] / (__expf(-w[e]) + 1.f);
                    auto put = [&](uint32_t part, uint16_t v) { *reinterpret_cast<uint16_t *>(a.ff + short_act_offset(f / 32, tok0 + e, slot >> 3, T, part) + (slot & 7) * 2) = v; };
                    if constexpr (EXACT) {
                        uint32_t b[3];
                        short_cut(b, y);
#pragma unroll
                        for (int i = 0; i < 3; i++) put(i, (uint16_t)(b[i] >> 16));
                    } else {
                        const uint16_t h = float_to_half_bits(y);
                        put(0, h);
                        put(1, float_to_half_bits(y - half_bits_to_float(h)));
                    }
                }
                continue;
            }
            const uint32_t z = tile / a.tiles_m, m = tile % a.tiles_m * 16 + r16;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t tok = tok0 + e;
                if (tok >= a.n) continue;
                if (EXACT && a.mode == kShortResidual) st_dev(out + (size_t)tok * a.ldo + m, v[e]);
                else if (z == 0) out[(size_t)tok * a.ldo + m] = v[e];
                else if (row_at + tok < a.backlog) a.cache[z - 1][(size_t)(row_at + tok) * a.ldo + m] = float_to_half_bits(v[e]);
            }
        }
    }
    if constexpr (EXACT) {
        if (a.mode != kShortResidual) return;
        // As in attention_kernel: write-through stores, acknowledged, then counted in; the last one reads with device-scope loads.  One
        // slice: the workgroup is its own last one.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (gridDim.y > 1) {
            if (threadIdx.x == 0) arrived = __hip_atomic_fetch_add(&a.counters[blockIdx.x], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
            if (arrived != gridDim.y - 1) return;
            if (threadIdx.x == 0) a.counters[blockIdx.x] = 0u;
        }
        constexpr int ROWS = RT * 16;
        static_assert(2 * kShortExact * ROWS <= sizeof red / 4, "x and x w of a row group");
        float *const xl = red, *const yl = red + kShortExact * ROWS;      // [token][row]
        const uint32_t row0 = tile0 * 16, rows = min((uint32_t)ROWS, a.ldo - row0);
        for (uint32_t i = threadIdx.x; i < a.n * ROWS; i += kShortWaves * 64) {
            const uint32_t tok = i / ROWS, r = i % ROWS;
            if (r >= rows) continue;
            const size_t at = (size_t)tok * a.ldo + row0 + r;
            uint32_t p[kShortSlices];
#pragma unroll
            for (int q = 0; q < kShortSlices; q++)
                if (q < (int)gridDim.y) p[q] = ld_dev(reinterpret_cast<const uint32_t *>(a.out[q] + at));
            const float x0 = a.res[at], w = a.norm_w[row0 + r];
            float t = __uint_as_float(p[0]);
#pragma unroll
            for (int q = 1; q < kShortSlices; q++)
                if (q < (int)gridDim.y) t += __uint_as_float(p[q]);
            t += x0;
            a.res[at] = t;
            xl[tok * ROWS + r] = t;
            yl[tok * ROWS + r] = t * w;
        }
        __syncthreads();
        for (uint32_t tok = wave; tok < a.n; tok += kShortWaves) {
            constexpr int PER = (ROWS + 63) / 64;
            float v[PER], sum = 0.f, q = 0.f;
#pragma unroll
            for (int j = 0; j < PER; j++) {
                v[j] = j * 64 + lane < (int)rows ? xl[tok * ROWS + j * 64 + lane] : 0.f;
                sum += v[j];
            }
            sum = wave_sum(sum);
            const float mean = sum / (float)rows;
#pragma unroll
            for (int j = 0; j < PER; j++)
                if (j * 64 + lane < (int)rows) q = fmaf(v[j] - mean, v[j] - mean, q);
            q = wave_sum(q);
            if (lane == 0) a.stats_out[blockIdx.x * kShortExact + tok] = make_float2(sum, q);
        }
        for (uint32_t i = threadIdx.x; i < a.n * (ROWS / 8); i += kShortWaves * 64) {
            const uint32_t tok = i / (ROWS / 8), r = i % (ROWS / 8) * 8, k = row0 + r;
            if (r >= rows) continue;
            const float4 *y = reinterpret_cast<const float4 *>(yl + tok * ROWS + r);
            float f[8];
            short_order<QT>(f, y[0], y[1], true);
            short_put(a.act_out, k / 32, tok, k % 32 / 8, T, f);
        }
    }
}

// x += the K slices of the product before, then normalize(x) * w (normalize.comp:34-64) as the next product's activations, halves
// scaled per token as in gemm_row_scale: in steps of 17 tokens and more, and in front of the first layer.  One workgroup per token, a
// thread per 8 elements (dim / 8 threads rounded up to whole waves;
// dim <= 8192, a multiple of 32): nothing but latency counts here, and a thread's loads are few and all in flight at once.
struct ShortNormArgs {
    float *x;
    const float *parts[kShortSlices];
    uint32_t nparts;
    const float *w;
    uint8_t *act;
    float *xscale;
    uint32_t dim, tiles;
};
template <int QT>
__global__ __launch_bounds__(1024) void short_norm_kernel(ShortNormArgs a)
{
    __shared__ float lds[48];
    const uint32_t row = blockIdx.x, i = threadIdx.x;
    const int wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const bool ok = i < a.dim / 8;
    const size_t ro = (size_t)row * a.dim;
    const uint32_t ic = ok ? i : 0, k[2] = {(ic >> 2) * 32 + (ic & 3) * 8, (ic >> 2) * 32 + (ic & 3) * 8 + 4};
    float4 x[2], w[2], p[kShortSlices][2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        w[h] = *reinterpret_cast<const float4 *>(a.w + k[h]);
        x[h] = *reinterpret_cast<const float4 *>(a.x + ro + k[h]);
#pragma unroll
        for (int q = 0; q < kShortSlices; q++)
            if (q < (int)a.nparts) p[q][h] = *reinterpret_cast<const float4 *>(a.parts[q] + ro + k[h]);
    }
    // the largest element of x w goes along with the sum: its exponent decides the row's scale, and 1 / rms multiplies every
    // element alike
    float s = 0.f, big = 0.f;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        if (a.nparts) {
            float4 t = p[0][h];
#pragma unroll
            for (int q = 1; q < kShortSlices; q++)
                if (q < (int)a.nparts) { t.x += p[q][h].x; t.y += p[q][h].y; t.z += p[q][h].z; t.w += p[q][h].w; }
            x[h].x = t.x + x[h].x; x[h].y = t.y + x[h].y; x[h].z = t.z + x[h].z; x[h].w = t.w + x[h].w;
            if (ok) *reinterpret_cast<float4 *>(a.x + ro + k[h]) = x[h];
        }
        if (!ok) x[h] = make_float4(0.f, 0.f, 0.f, 0.f);
        s += (x[h].x + x[h].y) + (x[h].z + x[h].w);
        big = fmaxf(big, fmaxf(fmaxf(fabsf(x[h].x * w[h].x), fabsf(x[h].y * w[h].y)), fmaxf(fabsf(x[h].z * w[h].z), fabsf(x[h].w * w[h].w))));
    }
    s = wave_sum(s);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) big = fmaxf(big, __shfl_xor(big, off, 64));
    if ((threadIdx.x & 63) == 0) { lds[wave] = s; lds[16 + wave] = big; }
    __syncthreads();
    s = 0.f;
    for (int v = 0; v < waves; v++) { s += lds[v]; big = fmaxf(big, lds[16 + v]); }
    const float mean = s / (float)a.dim;
    float q = 0.f;
    if (ok) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const float c0 = x[h].x - mean, c1 = x[h].y - mean, c2 = x[h].z - mean, c3 = x[h].w - mean;
            q = fmaf(c0, c0, q); q = fmaf(c1, c1, q); q = fmaf(c2, c2, q); q = fmaf(c3, c3, q);
        }
    }
    q = wave_sum(q);
    if ((threadIdx.x & 63) == 0) lds[32 + wave] = q;
    __syncthreads();
    q = 0.f;
    for (int v = 0; v < waves; v++) q += lds[32 + v];
    const float inv = rsqrtf(q / (float)a.dim);
    float up = 1.f;
    if (!short_exact(a.tiles)) {
        float down;
        up = gemm_row_scale(big * inv, &down);
        if (threadIdx.x == 0) a.xscale[row] = down;
    }
    if (!ok) return;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        x[h].x = (x[h].x * w[h].x) * inv; x[h].y = (x[h].y * w[h].y) * inv; x[h].z = (x[h].z * w[h].z) * inv; x[h].w = (x[h].w * w[h].w) * inv;
    }
    float f[8];
    short_order<QT>(f, x[0], x[1], short_exact(a.tiles));
#pragma unroll
    for (int e = 0; e < 8; e++) f[e] *= up;
    short_put(a.act, i >> 2, row, i & 3, a.tiles, f);
}

// Attention of 16 to 64 tokens: attention_batch_kernel's arithmetic, with the cache positions shared out over workgroups and the
// operand planes made on the way into LDS (a plane would be used once).  Without a running maximum the parts of a row are plain
// sums: numerators [split][n][H*R] and denominators [split][n][H], put together by short_attn_combine_kernel.  64 KB of LDS: two
// workgroups a CU.
struct ShortAttnArgs {
    const uint16_t *kcache, *vcache;   // [backlog][H*R] fp16, the batch's rows already in them
    const float *q;                    // [n][H*R]
    const float2 *trig_abs;            // [backlog][R/2]
    uint32_t pos0, n, heads, backlog;  // row z sits at pos0 + z
    uint32_t tiles_per_split;          // tiles of 64 positions
    float *num, *den;
    uint8_t *act;                      // the output projection's activations, `tiles` token tiles, or null: num and den are for short_attn_combine_kernel
    uint32_t *counters;                // short_attn_exact_kernel: one a head, zero before and after
    uint32_t tiles, q8;
};
// grid (heads, splits)
template <int R>
__global__ __launch_bounds__(256, 2) void short_attn_kernel(ShortAttnArgs a)
{
    constexpr int TK = kAttnBatchK;
    constexpr int KS = R / 16, DT = R / 32, C8 = R / 8;
    constexpr int PLANE = TK * R * 2;
    constexpr int XS = R + 4;
    static_assert(64 * XS * 4 <= 4 * PLANE, "the result exchange reuses the tile buffers");
    extern __shared__ __attribute__((aligned(16))) uint8_t short_lds[];      // kh, kl, v1, v2: 512 R bytes
    __shared__ float den_s[2][32];
    const uint32_t h = blockIdx.x, H = a.heads, D = H * R;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int qt = wave & 1, pt = wave >> 1, n32 = lane & 31, hh = lane >> 5;
    const uint32_t rows = min(a.pos0 + a.n, a.backlog);               // positions that hold data
    const uint32_t tile_end = min((blockIdx.y + 1) * a.tiles_per_split, (rows + TK - 1) / TK);

    // A tile's rows, requested a tile ahead.  K: thread t takes the 16-byte chunk t % C8 of rows t / C8, + 256 / C8, ...  V: two
    // dims (4 bytes) of eight positions, whose slots are a 16-byte chunk of either dim's row in the transposed planes.
    constexpr int PT = C8 * TK / 256, VT = R / 2 * 8 < 256 ? 1 : R / 2 * 8 / 256;     // R 32: half of the threads
    uint4 kq[PT];
    uint32_t vq[VT][8];
    auto vpos = [](int c8, int e) { return ((8 * c8 + e) & ~15) + attn_slot_pos((8 * c8 + e) & 15); };
    auto fetch = [&](uint32_t it) {
#pragma unroll
        for (int i = 0; i < PT; i++) {
            const uint32_t c = t + i * 256, p = min(it * TK + c / C8, rows - 1);
            kq[i] = *reinterpret_cast<const uint4 *>(a.kcache + (size_t)p * D + (size_t)h * R + c % C8 * 8);
        }
#pragma unroll
        for (int i = 0; i < VT; i++) {
            const uint32_t u = t + i * 256, dp = u % (R / 2), c8 = min(u / (R / 2), 7u);
#pragma unroll
            for (int e = 0; e < 8; e++)
                vq[i][e] = *reinterpret_cast<const uint32_t *>(a.vcache + (size_t)min(it * TK + vpos(c8, e), rows - 1) * D + (size_t)h * R + dp * 2);
        }
    };
    fetch(blockIdx.y * a.tiles_per_split);

    lv_h8 qh[KS], ql[KS];
    const uint32_t zq = 32 * qt + n32;
    const bool zok = zq < a.n;
    {
        const uint32_t pq = min(a.pos0 + zq, a.backlog - 1);
        const float *qr = a.q + (size_t)(zok ? zq : 0) * D + (size_t)h * R;
        const float2 *tr = a.trig_abs + (size_t)pq * (R / 2);
#pragma unroll
        for (int j = 0; j < KS; j++) {
            const float4 q0 = *reinterpret_cast<const float4 *>(qr + 16 * j + 8 * hh), q1 = *reinterpret_cast<const float4 *>(qr + 16 * j + 8 * hh + 4);
            const float4 c0 = *reinterpret_cast<const float4 *>(tr + 8 * j + 4 * hh), c1 = *reinterpret_cast<const float4 *>(tr + 8 * j + 4 * hh + 2);
            float f[8] = {q0.x * c0.x - q0.y * c0.y, q0.x * c0.y + q0.y * c0.x, q0.z * c0.z - q0.w * c0.w, q0.z * c0.w + q0.w * c0.z,
                          q1.x * c1.x - q1.y * c1.y, q1.x * c1.y + q1.y * c1.x, q1.z * c1.z - q1.w * c1.w, q1.z * c1.w + q1.w * c1.z};
            if (!zok) {
#pragma unroll
                for (int e = 0; e < 8; e++) f[e] = 0.f;
            }
            uint4 hi, lo;
            gemm_split8(hi, lo, f);
            qh[j] = __builtin_bit_cast(lv_h8, hi);
            ql[j] = __builtin_bit_cast(lv_h8, lo);
        }
    }
    const float scale = rsqrtf((float)R);
    lv_f16v acc[DT];
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[d][r] = 0.f;
    float den = 0.f;
    const uint32_t limit = a.pos0 + zq;
    const bool tile_live = 32 * qt < (int)a.n;                        // this wave's 32 queries hold one of the batch
    const uint32_t wave_last = a.pos0 + min(32u * qt + 31, a.n - 1);

    for (uint32_t it = blockIdx.y * a.tiles_per_split; it < tile_end; it++) {
        const uint32_t k0 = it * TK;
        __syncthreads();                                              // the tile before is consumed
#pragma unroll
        for (int i = 0; i < PT; i++) {
            const int c = t + i * 256, c8 = c % C8, row = c / C8;
            const uint32_t p = k0 + row;
            float f[8];
            const bool live = p < rows;                               // rows past the data: zeros, which the masked sums can take
            const float4 cs0 = *reinterpret_cast<const float4 *>(a.trig_abs + (size_t)min(p, rows - 1) * (R / 2) + c8 * 4);
            const float4 cs1 = *reinterpret_cast<const float4 *>(a.trig_abs + (size_t)min(p, rows - 1) * (R / 2) + c8 * 4 + 2);
            const uint32_t kw[4] = {kq[i].x, kq[i].y, kq[i].z, kq[i].w};
            const float cc[4] = {cs0.x, cs0.z, cs1.x, cs1.z}, ss[4] = {cs0.y, cs0.w, cs1.y, cs1.w};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float x = half_bits_to_float((uint16_t)(kw[j] & 0xffffu)), y = half_bits_to_float((uint16_t)(kw[j] >> 16));
                f[2 * j] = live ? x * cc[j] - y * ss[j] : 0.f;
                f[2 * j + 1] = live ? x * ss[j] + y * cc[j] : 0.f;
            }
            uint4 hi, lo;
            gemm_split8(hi, lo, f);
            uint8_t *kd = short_lds + row * 2 * R + (c8 ^ attn_kswz<R>(row)) * 16;
            *reinterpret_cast<uint4 *>(kd) = hi;
            *reinterpret_cast<uint4 *>(kd + PLANE) = lo;
        }
#pragma unroll
        for (int i = 0; i < VT; i++) {
            const int u = t + i * 256, dp = u % (R / 2), c8 = u / (R / 2);
            if (R < 64 && c8 >= 8) break;
#pragma unroll
            for (int half = 0; half < 2; half++) {
                uint32_t w1[4], w2[4];
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    uint32_t b1[2], b2[2];
#pragma unroll
                    for (int x = 0; x < 2; x++) {
                        const bool live = k0 + vpos(c8, e + x) < rows;
                        const float v = live ? half_bits_to_float((uint16_t)(vq[i][e + x] >> (16 * half))) : 0.f;
                        b1[x] = __float_as_uint(v) & 0xffff0000u;
                        b2[x] = __float_as_uint(v - __uint_as_float(b1[x]));
                    }
                    w1[e / 2] = (b1[0] >> 16) | b1[1];
                    w2[e / 2] = (b2[0] >> 16) | (b2[1] & 0xffff0000u);
                }
                const int dim = 2 * dp + half;
                uint8_t *vd = short_lds + 2 * PLANE + dim * 128 + (c8 ^ (dim & 7)) * 16;
                *reinterpret_cast<uint4 *>(vd) = make_uint4(w1[0], w1[1], w1[2], w1[3]);
                *reinterpret_cast<uint4 *>(vd + PLANE) = make_uint4(w2[0], w2[1], w2[2], w2[3]);
            }
        }
        if (it + 1 < tile_end) fetch(it + 1);
        __syncthreads();
        if (!tile_live || k0 + 32 * pt > wave_last) continue;         // every pair of this wave's 32 x 32 tile is masked
        const uint8_t *kb = short_lds, *vb = kb + 2 * PLANE;
        lv_f16v sc;
#pragma unroll
        for (int r = 0; r < 16; r++) sc[r] = 0.f;
        {
            const int row = 32 * pt + n32;
            const uint8_t *kr = kb + row * 2 * R;
            const int sw = attn_kswz<R>(row);
#pragma unroll
            for (int j = 0; j < KS; j++) {
                const int c = (2 * j + hh) ^ sw;
                const lv_h8 ah = *reinterpret_cast<const lv_h8 *>(kr + c * 16), al = *reinterpret_cast<const lv_h8 *>(kr + PLANE + c * 16);
                sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, ql[j], sc, 0, 0, 0);
                sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, qh[j], sc, 0, 0, 0);
                sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, qh[j], sc, 0, 0, 0);
            }
        }
        // register r of sc: position k0 + 32 pt + 8 (r / 4) + 4 hh + r % 4, query n32 of the wave's tile
#pragma unroll
        for (int tt = 0; tt < 2; tt++) {
            uint32_t w1[4], w2[4], w3[4];
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                uint32_t b1[2], b2[2], b3[2];
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const int r = 8 * tt + e + u;
                    const uint32_t p = k0 + 32 * pt + 8 * (r / 4) + 4 * hh + (r % 4);
                    const bool ok = zok && p <= limit && p < a.backlog;
                    float e0 = __expf(sc[r] * scale);
                    e0 = ok ? e0 : 0.f;
                    den += e0;
                    b1[u] = __float_as_uint(e0) & 0xffff0000u;
                    const float r1 = e0 - __uint_as_float(b1[u]);
                    b2[u] = __float_as_uint(r1) & 0xffff0000u;
                    b3[u] = __float_as_uint(r1 - __uint_as_float(b2[u]));
                }
                w1[e / 2] = (b1[0] >> 16) | b1[1];
                w2[e / 2] = (b2[0] >> 16) | b2[1];
                w3[e / 2] = (b3[0] >> 16) | (b3[1] & 0xffff0000u);
            }
            const lv_b8 p1 = __builtin_bit_cast(lv_b8, make_uint4(w1[0], w1[1], w1[2], w1[3]));
            const lv_b8 p2 = __builtin_bit_cast(lv_b8, make_uint4(w2[0], w2[1], w2[2], w2[3]));
            const lv_b8 p3 = __builtin_bit_cast(lv_b8, make_uint4(w3[0], w3[1], w3[2], w3[3]));
#pragma unroll
            for (int d = 0; d < DT; d++) {
                const int dim = 32 * d + n32, c = (4 * pt + 2 * tt + hh) ^ (dim & 7);
                const lv_b8 va = *reinterpret_cast<const lv_b8 *>(vb + dim * 128 + c * 16);
                const lv_b8 vc = *reinterpret_cast<const lv_b8 *>(vb + PLANE + dim * 128 + c * 16);
                acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(p3, va, acc[d], 0, 0, 0);
                acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(p2, vc, acc[d], 0, 0, 0);
                acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(p2, va, acc[d], 0, 0, 0);
                acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(p1, vc, acc[d], 0, 0, 0);
                acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(p1, va, acc[d], 0, 0, 0);
            }
        }
    }
    // ---- the second position tile's sums to the first's waves, then out ---------------------------------------------------------
    den += __shfl_xor(den, 32, kWave);
    float *xch = reinterpret_cast<float *>(short_lds);
    __syncthreads();
    if (pt == 1) {
        if (hh == 0) den_s[qt][n32] = den;
#pragma unroll
        for (int d = 0; d < DT; d++)
#pragma unroll
            for (int r = 0; r < 16; r++) xch[(32 * qt + 8 * (r / 4) + 4 * hh + (r % 4)) * XS + 32 * d + n32] = acc[d][r];
    }
    __syncthreads();
    if (a.act) {
        if (pt == 0) {
            if (hh == 0) den_s[qt][n32] += den;
#pragma unroll
            for (int d = 0; d < DT; d++)
#pragma unroll
                for (int r = 0; r < 16; r++) xch[(32 * qt + 8 * (r / 4) + 4 * hh + (r % 4)) * XS + 32 * d + n32] += acc[d][r];
        }
        __syncthreads();
        for (uint32_t i = t; i < a.n * C8; i += 256) {
            const uint32_t z = i / C8, c = i % C8, k = h * R + (c >> 2) * 32, g = c & 3;
            const float *row = xch + z * XS + (c >> 2) * 32;
            const float total = den_s[z >> 5][z & 31];
            float4 va = *reinterpret_cast<const float4 *>(row + 8 * g);
            float4 vb = *reinterpret_cast<const float4 *>(row + 8 * g + 4);
            va.x /= total; va.y /= total; va.z /= total; va.w /= total;
            vb.x /= total; vb.y /= total; vb.z /= total; vb.w /= total;
            float f[8];
            if (a.q8 || !short_exact(a.tiles)) short_order<8>(f, va, vb, false);
            else short_order<4>(f, va, vb, true);
            short_put(a.act, k / 32, z, g, a.tiles, f);
        }
        return;
    }
    if (pt == 1) return;
    const size_t part = (size_t)blockIdx.y * a.n;
    if (hh == 0 && zok) a.den[(part + zq) * H + h] = den + den_s[qt][n32];
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const uint32_t z = 32 * qt + 8 * (r / 4) + 4 * hh + (r % 4);
            if (z < a.n) a.num[(part + z) * D + (size_t)h * R + 32 * d + n32] = acc[d][r] + xch[z * XS + 32 * d + n32];
        }
}

__device__ __forceinline__ void short_act_row(const ShortAttnArgs &a, uint32_t k, uint32_t z, float4 va, float4 vb, float den)
{
    va.x /= den; va.y /= den; va.z /= den; va.w /= den;
    vb.x /= den; vb.y /= den; vb.z /= den; vb.w /= den;
    float f[8];
    if (a.q8) short_order<8>(f, va, vb, short_exact(a.tiles));
    else short_order<4>(f, va, vb, short_exact(a.tiles));
    short_put(a.act, k / 32, z, k % 32 / 8, a.tiles, f);
}
// The end of a workgroup that has written its split of head h through to memory: the last of a head's splits to arrive adds them up, in their
// order, and makes the output projection's operands of them.  short_attn_combine_kernel in its place: us of 8 layers of 7B q8_0, 4 tokens behind 1000
// rows 668 and 651 so, 8 behind 300 645 and 635, 15 behind 1900 787 and 779; 13B q4_0, 8 behind 1500 731 and 721.  With more tokens a head
// is too much for one workgroup (17 behind 150 844 and 850, 45 behind 619 1042 and 1077, 64 behind 1900 1249 and 1306).
template <int R> __device__ __forceinline__ void short_attn_last(const ShortAttnArgs &a, uint32_t h)
{
    __shared__ uint32_t arrived;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) arrived = __hip_atomic_fetch_add(&a.counters[h], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (arrived != gridDim.y - 1) return;
    if (threadIdx.x == 0) a.counters[h] = 0u;
    const uint32_t D = a.heads * R;
    for (uint32_t i = threadIdx.x; i < a.n * (R / 8); i += 256) {
        const uint32_t z = i / (R / 8), k = h * R + i % (R / 8) * 8;
        float4 va = make_float4(0.f, 0.f, 0.f, 0.f), vb = va;
        float den = 0.f;
#pragma unroll 4
        for (uint32_t s = 0; s < gridDim.y; s++) {
            const size_t part = (size_t)s * a.n + z;
            const uint64_t *p = reinterpret_cast<const uint64_t *>(a.num + part * D + k);
            float2 v[4];
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = __builtin_bit_cast(float2, __hip_atomic_load(p + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
            den += __uint_as_float(ld_dev(reinterpret_cast<const uint32_t *>(a.den + part * a.heads + h)));
            va.x += v[0].x; va.y += v[0].y; va.z += v[1].x; va.w += v[1].y;
            vb.x += v[2].x; vb.y += v[2].y; vb.z += v[3].x; vb.w += v[3].y;
        }
        short_act_row(a, k, z, va, vb, den);
    }
}

// Attention of 2 to 15 tokens: fp32 throughout, on the fp32 matrix instruction, whose 16 columns are the step's queries.  attention_kernel
// reads a head's cache rows and rotations again for every query (15 queries behind 1900 positions: 0.9 GB through the L2s); here they are read
// once, rotated in registers and multiplied with all queries, 64 instructions per 16 positions whatever n is.  A layer of 7B, us with what makes
// the output projection's operands of it: 15 queries behind 1900 positions 65 and 25, 8 at the start of a sequence 10 and 7.
// Rotation by absolute positions; tiles, splits, num, den and act as short_attn_kernel.  A wave takes 16 of a tile's 64 positions; nothing is exchanged before the end:
//   scores    A = K (row: position l % 16), B = q (column: query l % 16), step j contracts dims g R/4 + j of the four lane groups g = l / 16
//   weighted  the result's register r holds position 4 g + r, which is how B = weights is wanted; A = V, rows m of tile t being dim m R/16 + t
template <int R>
__global__ __launch_bounds__(256, 2) void short_attn_exact_kernel(ShortAttnArgs a)
{
    constexpr int TK = kAttnBatchK;
    constexpr int KL = R / 4, VD = R / 16, C8 = R / 8, XS = R + 4;
    __shared__ __attribute__((aligned(16))) float xch[4 * 16 * XS];
    __shared__ float den_s[4][16];
    const uint32_t h = blockIdx.x, H = a.heads, D = H * R;
    const int t = threadIdx.x, lane = t & 63, l16 = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t rows = min(a.pos0 + a.n, a.backlog);               // positions that hold data
    const uint32_t tile_end = min((blockIdx.y + 1) * a.tiles_per_split, (rows + TK - 1) / TK);

    uint4 kq[KL / 8];
    float4 cs[KL / 4];
    uint32_t vq[4][VD / 2];
    auto fetch = [&](uint32_t base) {                                 // past the data: the last row again, masked below
        const uint32_t p = min(base + l16, rows - 1);
#pragma unroll
        for (int i = 0; i < KL / 8; i++) kq[i] = *reinterpret_cast<const uint4 *>(a.kcache + (size_t)p * D + (size_t)h * R + g * KL + i * 8);
#pragma unroll
        for (int i = 0; i < KL / 4; i++) cs[i] = *reinterpret_cast<const float4 *>(a.trig_abs + (size_t)p * (R / 2) + g * (KL / 2) + i * 2);
#pragma unroll
        for (int r = 0; r < 4; r++)
            __builtin_memcpy(vq[r], __builtin_assume_aligned(a.vcache + (size_t)min(base + 4 * g + r, rows - 1) * D + (size_t)h * R + l16 * VD, VD * 2), VD * 2);
    };
    fetch(blockIdx.y * a.tiles_per_split * TK + 16 * wave);

    const bool zok = (uint32_t)l16 < a.n;
    const uint32_t limit = a.pos0 + l16;                              // the last position query l16 sees
    float q[KL];
    {
        const float *qr = a.q + (size_t)(zok ? l16 : 0) * D + (size_t)h * R + g * KL;
        const float2 *tr = a.trig_abs + (size_t)min(limit, a.backlog - 1) * (R / 2) + g * (KL / 2);
#pragma unroll
        for (int i = 0; i < KL / 4; i++) {
            const float4 x = *reinterpret_cast<const float4 *>(qr + i * 4), c = *reinterpret_cast<const float4 *>(tr + i * 2);
            q[4 * i] = zok ? x.x * c.x - x.y * c.y : 0.f;
            q[4 * i + 1] = zok ? x.x * c.y + x.y * c.x : 0.f;
            q[4 * i + 2] = zok ? x.z * c.z - x.w * c.w : 0.f;
            q[4 * i + 3] = zok ? x.z * c.w + x.w * c.z : 0.f;
        }
    }
    const float scale = rsqrtf((float)R);
    lv_f4v acc[VD];
#pragma unroll
    for (int d = 0; d < VD; d++) acc[d] = lv_f4v{0.f, 0.f, 0.f, 0.f};
    float den = 0.f;

    for (uint32_t it = blockIdx.y * a.tiles_per_split; it < tile_end; it++) {
        const uint32_t base = it * TK + 16 * wave;
        if (base >= rows) break;
        float k[KL];
#pragma unroll
        for (int i = 0; i < KL / 4; i++) {
            const uint32_t w0 = i & 1 ? kq[i / 2].z : kq[i / 2].x, w1 = i & 1 ? kq[i / 2].w : kq[i / 2].y;
            const float x0 = half_bits_to_float((uint16_t)w0), y0 = half_bits_to_float((uint16_t)(w0 >> 16));
            const float x1 = half_bits_to_float((uint16_t)w1), y1 = half_bits_to_float((uint16_t)(w1 >> 16));
            k[4 * i] = x0 * cs[i].x - y0 * cs[i].y;
            k[4 * i + 1] = x0 * cs[i].y + y0 * cs[i].x;
            k[4 * i + 2] = x1 * cs[i].z - y1 * cs[i].w;
            k[4 * i + 3] = x1 * cs[i].w + y1 * cs[i].z;
        }
        uint32_t v[4][VD / 2];
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int i = 0; i < VD / 2; i++) v[r][i] = vq[r][i];
        if (it + 1 < tile_end) fetch(base + TK);
        lv_f4v sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < KL; j++) sc = __builtin_amdgcn_mfma_f32_16x16x4f32(k[j], q[j], sc, 0, 0, 0);
        float e[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const uint32_t p = base + 4 * g + r;
            const float w = __expf(sc[r] * scale);
            e[r] = zok && p <= limit && p < rows ? w : 0.f;
            den += e[r];
        }
        if (base + 15 > a.pos0) {
            // Rows that some queries do not see.  A weight of zero times an infinity or a NaN of such a row would reach them: these values
            // are left to the queries that see them.
            auto wild = [](uint32_t half) { return (half & 0x7c00u) == 0x7c00u; };
            bool any = false;
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int i = 0; i < VD / 2; i++) {
                    const bool lo = wild(v[r][i]), hi = wild(v[r][i] >> 16);
                    any |= lo || hi;
                    v[r][i] &= (lo ? 0u : 0xffffu) | (hi ? 0u : 0xffff0000u);
                }
            if (__any(any)) {
#pragma unroll
                for (int m = 0; m < 16; m++) {
                    const uint32_t p = base + m;
                    const float w = __shfl(e[m & 3], (m >> 2) * 16 + l16, kWave);
                    const uint16_t *vr = a.vcache + (size_t)min(p, rows - 1) * D + (size_t)h * R + 4 * g * VD;
                    if (!zok || p > limit || p >= rows) continue;
#pragma unroll
                    for (int i = 0; i < 4 * VD; i++)
                        if (wild(vr[i])) acc[i % VD][i / VD] = fmaf(w, half_bits_to_float(vr[i]), acc[i % VD][i / VD]);
                }
            }
        }
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int d = 0; d < VD; d++)
                acc[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(half_bits_to_float((uint16_t)(v[r][d / 2] >> (16 * (d & 1)))), e[r], acc[d], 0, 0, 0);
    }
    // acc[d][r]: dim (4 g + r) VD + d of query l16.  The waves' sums, then out
    den += __shfl_xor(den, 16, kWave);
    den += __shfl_xor(den, 32, kWave);
    if (g == 0) den_s[wave][l16] = den;
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
        for (int d = 0; d < VD; d++) xch[(wave * 16 + l16) * XS + (4 * g + r) * VD + d] = acc[d][r];
    __syncthreads();
    auto total = [&](uint32_t z, uint32_t d) {
        float4 s = *reinterpret_cast<const float4 *>(xch + z * XS + d);
#pragma unroll
        for (int w = 1; w < 4; w++) {
            const float4 x = *reinterpret_cast<const float4 *>(xch + (w * 16 + z) * XS + d);
            s.x += x.x; s.y += x.y; s.z += x.z; s.w += x.w;
        }
        return s;
    };
    auto weight = [&](uint32_t z) { return (den_s[0][z] + den_s[1][z]) + (den_s[2][z] + den_s[3][z]); };
    if (gridDim.y == 1) {
        for (uint32_t i = t; i < a.n * C8; i += 256) {
            const uint32_t z = i / C8, d = i % C8 * 8;
            short_act_row(a, h * R + d, z, total(z, d), total(z, d + 4), weight(z));
        }
        return;
    }
    const size_t part = (size_t)blockIdx.y * a.n;
    for (uint32_t i = t; i < a.n * (R / 4); i += 256) {
        const uint32_t z = i / (R / 4), d = i % (R / 4) * 4;
        const float4 s = total(z, d);
        uint64_t *p = reinterpret_cast<uint64_t *>(a.num + (part + z) * D + (size_t)h * R + d);
        __hip_atomic_store(p, __builtin_bit_cast(uint64_t, make_float2(s.x, s.y)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(p + 1, __builtin_bit_cast(uint64_t, make_float2(s.z, s.w)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if ((uint32_t)t < a.n) st_dev(a.den + (part + t) * H + h, weight(t));
    if (a.act) short_attn_last<R>(a, h);
}

// numerators and denominators of all splits, in order -> the output projection's activations.  grid (D / 8 / 256 rounded up, n)
struct ShortCombineArgs {
    const float *num, *den;
    uint32_t splits, n, heads, rot, tiles;
    uint8_t *act;
};
template <int QT>
__global__ __launch_bounds__(256) void short_attn_combine_kernel(ShortCombineArgs a)
{
    const uint32_t D = a.heads * a.rot, i = blockIdx.x * 256 + threadIdx.x, z = blockIdx.y;
    if (i >= D / 8) return;
    const uint32_t ka = (i >> 2) * 32 + (i & 3) * 8, kb = (i >> 2) * 32 + (i & 3) * 8 + 4;
    const uint32_t h = ka / a.rot;                     // a block of 32 lies in one head
    float4 va = make_float4(0.f, 0.f, 0.f, 0.f), vb = va;
    float den = 0.f;
    for (uint32_t s = 0; s < a.splits; s++) {
        const size_t part = (size_t)s * a.n + z;
        const float4 pa = *reinterpret_cast<const float4 *>(a.num + part * D + ka), pb = *reinterpret_cast<const float4 *>(a.num + part * D + kb);
        va.x += pa.x; va.y += pa.y; va.z += pa.z; va.w += pa.w;
        vb.x += pb.x; vb.y += pb.y; vb.z += pb.z; vb.w += pb.w;
        den += a.den[part * a.heads + h];
    }
    va.x /= den; va.y /= den; va.z /= den; va.w /= den;
    vb.x /= den; vb.y /= den; vb.z /= den; vb.w /= den;
    float f[8];
    short_order<QT>(f, va, vb, short_exact(a.tiles));
    short_put(a.act, i >> 2, z, i & 3, a.tiles, f);
}

}  // namespace lv
