// lv_small.h — one token of a small model as one launch (gfx950).
//
// What bounds a token of a model of a few hundred columns is neither bytes nor arithmetic: at width 256, 2 layers, the operator chain is
// 24 dependent launches of 1 to 8 us, 117 us a token of which less than 1 us is bytes.  Here a few workgroups (small_wgs: about one pair
// of tiles a wave in the feed-forward) stay for the whole token and hand vectors to each other as the persistent kernel of the large
// shapes does (lv_mega.h: the data is the flag, every wait is bounded), with sizes known at run time and the operator chain's weights:
//
//   per layer: a workgroup a head forms its query, key and value rows and attends, all inside the workgroup -> o
//              all workgroups: x += Wo o -> x1; norm, gate and up -> ff; x1 += W2 ff -> x2
//
// With partial sums, two hand-overs a layer instead of four: a head's workgroup multiplies its own o by its columns of Wo, a workgroup its
// own blocks of ff by their columns of W2, and every reader adds the parts up.  More values are handed over, (heads + workgroups) D a
// layer: for narrow models only (lv_small_plan.h).
//
// Width 256, 2 layers: 53.6 us a token with four hand-overs a layer, 18.7 of them a layer; 47.9 with two, 14.2.
// A wave takes tiles of 64 blocks: L lanes a row (a power of two, 8 to 64), 64 / L rows; the first kSmallDepth tiles of a phase are
// asked for before the vector they are multiplied with is waited for.
#pragma once

#include "lv_kernels.h"
#include "lv_mega.h"
#include "lv_small_plan.h"

namespace lv {

constexpr int kSmallDepth = 4;             // tiles in flight a wave

struct SmallLayer {
    MatView wq, wk, wv, wo, w1, w2, w3;
    const float *attn_norm, *ffn_norm;
};

struct SmallArgs {
    const SmallLayer *layer;
    MatView output;
    const float *norm;
    MatView tok;               // quantised embedding table ...
    const float *tok_f32;      // ... or the fp32 one (then not null)
    int tok_q4;
    uint16_t *kv;              // [layers][2][backlog][D]
    const float2 *trig;        // [backlog][R / 2]
    float *xchg, *xchg_rearm;  // [layers][o D, x1 D, ff F, x2 D], all kNotReady; the other set is made so during this token
    float *logits, *logits_host;   // on the device and in pinned memory: no launch of its own copies them
    uint32_t *status;
    uint32_t layers, vocab, backlog, pos, token, D, F, heads, spin_limit;
    uint32_t own;              // 0, or with partial sums: feed-forward blocks of a workgroup, a power of two
};

// Pointers to weights are kept as addresses of global memory: loads through a pointer that itself came from memory would otherwise be
// ones that might go to LDS, which are waited for together with those.
typedef uint32_t small_u4 __attribute__((ext_vector_type(4)));
struct SmallView {
    const __attribute__((address_space(1))) small_u4 *codes;
    const __attribute__((address_space(1))) void *scales;      // fp16 or fp32
};
template <bool SF32>
__device__ __forceinline__ SmallView small_view(const void *codes, const uint16_t *scales, const float *scales_f32)
{
    return {(const __attribute__((address_space(1))) small_u4 *)codes, (const __attribute__((address_space(1))) void *)(SF32 ? (const void *)scales_f32 : scales)};
}
// an entry of the table, through the scalar cache: the kernel's own stores would otherwise make it a load a lane
typedef const __attribute__((address_space(4))) uint64_t *small_const_p;
template <bool SF32>
__device__ __forceinline__ SmallView small_view(const MatView *p)
{
    static_assert(sizeof(MatView) == 32, "codes, scales, rows and columns, fp32 scales");
    const small_const_p c = (small_const_p)p;
    return small_view<SF32>((const void *)c[0], (const uint16_t *)c[1], (const float *)c[3]);
}
typedef const __attribute__((address_space(1))) float *small_float_p;
__device__ __forceinline__ small_float_p small_norm(const float *const *p) { return (small_float_p)*(small_const_p)p; }

// Every exchanged float is polled until it is not kNotReady: a NaN of that pattern must not be stored
__device__ __forceinline__ void small_publish(float *p, float v) { st_dev(p, v == v ? v : __uint_as_float(0x7fc00000u)); }

template <int QT>
struct SmallRaw {
    small_u4 c, c2;
    uint32_t d;
};

// A product of one, two or three matrices over the same columns, dealt tile by tile to `waves` waves.  Rows are those of all three one
// behind the other, `part` of each from row row0 on (kSmallStacked), or tile t is tile t of the first and then tile t of the second
// matrix, whose results leave together (kSmallPair).  All phases of a token run through the one copy of this code: a line of code is
// fetched from memory by the workgroup that first gets there, which at this size takes longer than what the line does.
enum SmallKind { kSmallStacked, kSmallPair };

template <int QT, bool SF32>
struct SmallGemv {
    SmallView m0, m1, m2;
    uint32_t kind, nb, rows, part, row0, waves;
    int shift, lane;                     // lanes a row = 1 << shift
    uint32_t tile, ftile, fcol, fmat;    // next tile of this wave; what is fetched next
    uint32_t col, mat;
    float acc, first_sum;
    SmallRaw<QT> q[kSmallDepth];

    __device__ __forceinline__ uint32_t tile_rows() const { return 64u >> shift; }

    // without a branch (past the end block 0 is read): a value that may come from either side of one is waited for where the sides meet
    __device__ __forceinline__ void fetch(SmallRaw<QT> &t)
    {
        const uint32_t first = ftile * tile_rows();
        const uint32_t c = (fcol << shift) + (lane & ((1 << shift) - 1));
        const uint32_t r = first + (lane >> shift);
        // uniform: a tile never spans two matrices, and what is left of a matrix row by row is the last one's
        const uint32_t mi = kind == kSmallPair ? fmat : first >= 2 * part ? 2 : first >= part ? 1 : 0;
        const uint32_t at = kind == kSmallPair ? 0 : mi * part;
        // chosen among values: among members it would be a choice of addresses, and all of this would live in memory
        const auto c0 = m0.codes, c1 = m1.codes, c2 = m2.codes;
        const auto s0 = m0.scales, s1 = m1.scales, s2 = m2.scales;
        const auto codes = mi == 0 ? c0 : mi == 1 ? c1 : c2;
        const auto scales = mi == 0 ? s0 : mi == 1 ? s1 : s2;
        const uint32_t b = r < rows && c < nb ? (row0 + r - at) * nb + c : 0;
        if constexpr (QT == 4) t.c = codes[b];
        else { t.c = codes[2 * b]; t.c2 = codes[2 * b + 1]; }
        if constexpr (SF32) t.d = ((const __attribute__((address_space(1))) uint32_t *)scales)[b];
        else t.d = ((const __attribute__((address_space(1))) uint16_t *)scales)[b];
        const bool last = ((fcol + 1) << shift) >= nb, next = last && (kind != kSmallPair || fmat == 1);
        fcol = last ? 0 : fcol + 1;
        fmat = last && !next ? 1 : next ? 0 : fmat;
        ftile += next ? waves : 0;
    }
    __device__ __forceinline__ void start(uint32_t wave, uint32_t waves_, uint32_t nb_, uint32_t rows_)
    {
        lane = threadIdx.x & 63;
        nb = nb_; rows = rows_; waves = waves_;
        shift = small_lanes_log2(nb);
        tile = ftile = wave; fcol = fmat = col = mat = 0;
        acc = first_sum = 0.f;
#pragma unroll
        for (int j = 0; j < kSmallDepth; j++) fetch(q[j]);
    }
    __device__ __forceinline__ float row_total(float v) const
    {
        if (shift == 3) return group8_sum(v);
        if (shift == 4) return group16_sum(v);
        if (shift == 5) return half_wave_sum(v);
        return wave_sum(v);
    }
    template <class Emit>
    __device__ __forceinline__ void step(SmallRaw<QT> &t, const float *xs, Emit &&emit)
    {
        const int sub = lane & ((1 << shift) - 1);
        const uint32_t c = (col << shift) + sub;
        float xr[32], xsum;
        load_slab(xr, xsum, xs, (int)c, c < nb);
        const float d = SF32 ? __uint_as_float(t.d) : half_bits_to_float((uint16_t)t.d);
        const uint4 qa = make_uint4(t.c.x, t.c.y, t.c.z, t.c.w);
        float s;
        if constexpr (QT == 4) s = (q4_block_dot(qa, xr) - 8.f * xsum) * d;
        else s = (q8_block_dot(qa, make_uint4(t.c2.x, t.c2.y, t.c2.z, t.c2.w), xr) - 128.f * xsum) * d;
        acc += c < nb ? s : 0.f;
        fetch(t);
        if ((++col << shift) < nb) return;
        col = 0;
        const float total = row_total(acc);
        acc = 0.f;
        if (kind == kSmallPair && mat == 0) {
            mat = 1;
            first_sum = total;
            return;
        }
        mat = 0;
        const uint32_t r = tile * tile_rows() + (lane >> shift);
        if (sub == 0 && r < rows) emit(r, first_sum, total);
        tile += waves;
    }
    // xs: the vector in LDS (xs_index); emit(row, total of the pair's first matrix, total) by one lane a row
    template <class Emit>
    __device__ __forceinline__ void run(const float *xs, Emit &&emit)
    {
        static_assert(kSmallDepth == 4, "a step a place of the queue");
        // a place is refilled where it is used: moving the queue up would wait for what is on its way
        while (true) {
            if (tile * tile_rows() >= rows) return;
            step(q[0], xs, emit);
            if (tile * tile_rows() >= rows) return;
            step(q[1], xs, emit);
            if (tile * tile_rows() >= rows) return;
            step(q[2], xs, emit);
            if (tile * tile_rows() >= rows) return;
            step(q[3], xs, emit);
        }
    }
};

__device__ __forceinline__ float small_block_sum(float v, float *red)
{
    v = wave_sum(v);
    lds_barrier();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    lds_barrier();
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < kSmallWaves; i++) t += red[i];
    return t;
}

// the D values v of this thread (element threadIdx.x + j * kSmallThreads) into LDS: as they are and, with weights, normalised (normalize_kernel)
__device__ __forceinline__ void small_stage_x(const float (&v)[2], uint32_t D, small_float_p w, float *xraw, float *xs, float *red)
{
    float wv[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const uint32_t i = threadIdx.x + j * kSmallThreads;
        wv[j] = w && i < D ? w[i] : 0.f;
        if (i < D) xraw[i] = v[j];
    }
    if (!w) {
        lds_barrier();
        return;
    }
    const float mean = small_block_sum(v[0] + v[1], red) / (float)D;
    float q = 0.f;
#pragma unroll
    for (int j = 0; j < 2; j++)
        if (threadIdx.x + j * kSmallThreads < D) q = fmaf(v[j] - mean, v[j] - mean, q);
    const float inv = rsqrtf(small_block_sum(q, red) / (float)D);
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const uint32_t i = threadIdx.x + j * kSmallThreads;
        if (i < D) xs[xs_index(i)] = (v[j] * wv[j]) * inv;
    }
    lds_barrier();
}

__device__ __forceinline__ void small_poll_x(float (&v)[2], const float *src, uint32_t D, const SmallArgs &a)
{
    const bool want[2] = {threadIdx.x < D, threadIdx.x + kSmallThreads < D};
    poll_values<2>(v, src + threadIdx.x, kSmallThreads, want, a.status, a.spin_limit);
}

// a vector of n values, as it is, into LDS
__device__ __forceinline__ void small_stage(const float *src, uint32_t n, float *xs, const SmallArgs &a)
{
    lds_barrier();                   // other waves still read what is there
    for (uint32_t i0 = threadIdx.x; i0 < n; i0 += 4 * kSmallThreads) {
        float v[4];
        const bool want[4] = {true, i0 + kSmallThreads < n, i0 + 2 * kSmallThreads < n, i0 + 3 * kSmallThreads < n};
        poll_values<4>(v, src + i0, kSmallThreads, want, a.status, a.spin_limit);
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (want[j]) xs[xs_index(i0 + j * kSmallThreads)] = v[j];
    }
    lds_barrier();
}

// v += `count` vectors of D floats one behind the other (D a multiple of 4), in an order that hangs on D alone
__device__ __forceinline__ void small_add_parts(float (&v)[2], const float *src, uint32_t count, uint32_t D, float *sums, const SmallArgs &a)
{
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    constexpr int AHEAD = 4;
    const uint32_t quads = D / 4, groups = kSmallThreads / quads, grp = threadIdx.x / quads, q = threadIdx.x - grp * quads;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(src), 0, (int)(count * D * 4), 0x00020000);
    float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
    for (uint32_t p0 = grp; p0 < count && grp < groups; p0 += AHEAD * groups) {
        u4 u[AHEAD];
        uint32_t spins = 0;
        bool pending;
        do {
            pending = false;
            asm volatile("" ::: "memory");      // every turn issues the loads again; behind the last part they return zeros
#pragma unroll
            for (int j = 0; j < AHEAD; j++) {
                u[j] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)(((p0 + j * groups) * D + q * 4) * 4), 0, 16 /* device scope */);
                pending |= (u[j].x == kNotReady) | (u[j].y == kNotReady) | (u[j].z == kNotReady) | (u[j].w == kNotReady);
            }
        } while (pending && ++spins < a.spin_limit);
        if (pending) *a.status = 1u;
#pragma unroll
        for (int j = 0; j < AHEAD; j++) {
            t.x += __uint_as_float(u[j].x); t.y += __uint_as_float(u[j].y); t.z += __uint_as_float(u[j].z); t.w += __uint_as_float(u[j].w);
        }
    }
    lds_barrier();                   // other waves may still read the last sums
    if (grp < groups) *reinterpret_cast<float4 *>(sums + (grp * quads + q) * 4) = t;
    lds_barrier();
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const uint32_t i = threadIdx.x + j * kSmallThreads;
        if (i < D)
            for (uint32_t g = 0; g < groups; g++) v[j] += sums[g * D + i];
    }
}

// A workgroup's columns of a matrix of D rows of nb blocks: blocks c0 .. c0 + n - 1 of every row, `wide` (n rounded up to a power of two) lanes
// a row.  Asked for early, multiplied with a vector in LDS, the rows' sums published.
template <int QT, bool SF32>
struct SmallColumns {
    SmallRaw<QT> q[kSmallPartBlocks];

    __device__ __forceinline__ void fetch(const SmallView &m, uint32_t nb, uint32_t c0, uint32_t n, uint32_t wide, uint32_t D)
    {
#pragma unroll
        for (uint32_t j = 0; j < kSmallPartBlocks; j++) {
            const uint32_t i = threadIdx.x + j * kSmallThreads, r = i / wide, k = i - r * wide, b = r < D && k < n ? r * nb + c0 + k : 0;
            if constexpr (QT == 4) q[j].c = m.codes[b];
            else { q[j].c = m.codes[2 * b]; q[j].c2 = m.codes[2 * b + 1]; }
            if constexpr (SF32) q[j].d = ((const __attribute__((address_space(1))) uint32_t *)m.scales)[b];
            else q[j].d = ((const __attribute__((address_space(1))) uint16_t *)m.scales)[b];
        }
    }
    __device__ __forceinline__ void publish(const float *x, uint32_t n, uint32_t wide, uint32_t D, float *out)
    {
#pragma unroll
        for (uint32_t j = 0; j < kSmallPartBlocks; j++) {
            if (j * kSmallThreads >= D * wide) break;
            const uint32_t i = threadIdx.x + j * kSmallThreads, r = i / wide, k = i - r * wide;
            float xr[32], xsum = 0.f;
            const float4 *src = reinterpret_cast<const float4 *>(x + (k < n ? k : 0) * 32);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float4 f = src[e];
                xr[4 * e] = f.x; xr[4 * e + 1] = f.y; xr[4 * e + 2] = f.z; xr[4 * e + 3] = f.w;
                xsum += (f.x + f.y) + (f.z + f.w);
            }
            const float d = SF32 ? __uint_as_float(q[j].d) : half_bits_to_float((uint16_t)q[j].d);
            const uint4 qa = make_uint4(q[j].c.x, q[j].c.y, q[j].c.z, q[j].c.w);
            float s;
            if constexpr (QT == 4) s = (q4_block_dot(qa, xr) - 8.f * xsum) * d;
            else s = (q8_block_dot(qa, make_uint4(q[j].c2.x, q[j].c2.y, q[j].c2.z, q[j].c2.w), xr) - 128.f * xsum) * d;
            s = k < n ? s : 0.f;
            for (uint32_t off = 1; off < wide; off <<= 1) s += __shfl_xor(s, (int)off, kWave);
            if (k == 0 && r < D) small_publish(out + r, s);
        }
    }
};

// PARTS: with partial sums (args.own).  Instances of their own: the code of both ways in one made either 2 to 4 % slower (a line of code is
// fetched from memory; 768 wide, 12 layers with four hand-overs 378 -> 392 us).
template <int QT, bool SF32, int R, bool PARTS>
__global__ __launch_bounds__(kSmallThreads) void small_decode_kernel(SmallArgs a)
{
    constexpr int LPR = R / 8, RPB = kSmallThreads / LPR, BATCH = 2;     // lanes a cache row, rows of the workgroup at once, times BATCH
    __shared__ __align__(16) float xs[kSmallMaxFf];
    __shared__ __align__(16) float xraw[kSmallMaxDim];
    __shared__ __align__(16) float qs[R];
    __shared__ __align__(16) uint16_t knew[R], vnew[R];
    __shared__ float part[kSmallWaves][R + 1], red[kSmallWaves];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t D = a.D, F = a.F, nbD = D / 32, nbF = F / 32, G = gridDim.x, cur = a.pos;
    const uint32_t gw = blockIdx.x + wave * G, waves = G * kSmallWaves;   // consecutive tiles on different CUs
    const bool attends = blockIdx.x < a.heads;
    const uint32_t own = PARTS ? a.own : 0, per = small_layer_floats(D, F, a.heads, own);
    // with partial sums: this workgroup's feed-forward blocks
    const uint32_t parts = PARTS ? small_parts(F, own) : 0, c0 = blockIdx.x * own, nown = blockIdx.x < parts ? min(own, nbF - c0) : 0;
    float *const sums = xs;          // of parts, before xs is the norm

    for (uint32_t i = blockIdx.x * kSmallThreads + tid; i < a.layers * per; i += G * kSmallThreads) st_dev(a.xchg_rearm + i, __uint_as_float(kNotReady));

    float v[2] = {};
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const uint32_t i = tid + j * kSmallThreads;
        if (i >= D) continue;
        if (a.tok_f32) v[j] = a.tok_f32[(size_t)a.token * D + i];
        else {
            const uint64_t b = (uint64_t)a.token * nbD + i / 32;
            const uint32_t e = i % 32;
            const uint8_t *codes = reinterpret_cast<const uint8_t *>(a.tok.codes) + b * (a.tok_q4 ? 16 : 32);
            const int code = a.tok_q4 ? (int)((codes[e % 16] >> (e < 16 ? 0 : 4)) & 15) - 8 : (int)(int8_t)codes[e];
            v[j] = (float)code * mat_scale(a.tok, b);
        }
    }

    // phases of a layer: 0 a head's query, key, value and its attention, 1 Wo, 2 gate and up, 3 W2; behind the layers 4, the output matrix
    for (uint32_t step = 0; step <= 4 * a.layers; step++) {
        const uint32_t li = step / 4, ph = step == 4 * a.layers ? 4 : step % 4;
        const SmallLayer &l = a.layer[ph == 4 ? 0 : li];
        float *const o = a.xchg + (size_t)li * per, *const x1 = o + D, *const ff = x1 + D, *const x2 = ff + F;   // o - D: the layer before's x2
        if (ph == 0 && !attends) continue;
        if (PARTS && (ph == 1 || ph == 3)) continue;
        float *const part1 = o, *const part2 = o + a.heads * D;      // with partial sums; part1 - parts D: the layer before's part2

        SmallGemv<QT, SF32> g;
        g.kind = ph == 2 ? kSmallPair : kSmallStacked;
        g.m0 = ph == 4 ? small_view<SF32>(a.output.codes, a.output.scales, a.output.scales_f32) : small_view<SF32>(ph == 0 ? &l.wq : ph == 1 ? &l.wo : ph == 2 ? &l.w3 : &l.w2);
        g.m1 = g.m2 = g.m0;
        g.row0 = 0;
        g.part = 0x7fffffffu;
        if (ph == 0) {
            g.m1 = small_view<SF32>(&l.wk);
            g.m2 = small_view<SF32>(&l.wv);
            g.row0 = blockIdx.x * R;
            g.part = R;
        }
        if (ph == 2) g.m1 = small_view<SF32>(&l.w1);
        const bool mine = ph == 0 || (ph == 2 && PARTS);             // a product of this workgroup alone
        if (ph == 2 && PARTS) g.row0 = 32 * c0;
        g.start(mine ? wave : gw, mine ? kSmallWaves : waves, ph == 3 ? nbF : nbD, ph == 0 ? 3 * R : ph == 2 ? (PARTS ? 32 * nown : F) : ph == 4 ? a.vocab : D);
        SmallColumns<QT, SF32> cols;
        if constexpr (PARTS) {
            if (ph == 0) cols.fetch(small_view<SF32>(&l.wo), nbD, blockIdx.x * (R / 32), R / 32, R / 32, D);
            if (ph == 2) cols.fetch(small_view<SF32>(&l.w2), nbF, c0, nown, own, D);
        }

        // the first cache rows come on their way before anything is waited for; the new row is in LDS only
        uint16_t *const kc = a.kv + (size_t)(2 * li) * a.backlog * D + blockIdx.x * R, *const vc = kc + (size_t)a.backlog * D;
        const int sub = tid % LPR, rsel = tid / LPR;
        uint4 kr[BATCH], vr[BATCH];
        float4 t0[BATCH], t1[BATCH];
        const auto rows_at = [&](uint32_t p0) {
#pragma unroll
            for (int j = 0; j < BATCH; j++) {
                const uint32_t p = min(p0 + j * RPB + rsel, cur);
                if (p < cur) {
                    kr[j] = *reinterpret_cast<const uint4 *>(kc + (size_t)p * D + sub * 8);
                    vr[j] = *reinterpret_cast<const uint4 *>(vc + (size_t)p * D + sub * 8);
                }
                const float4 *tp = reinterpret_cast<const float4 *>(a.trig + (size_t)(cur - p) * (R / 2) + sub * 4);
                t0[j] = tp[0];
                t1[j] = tp[1];
            }
        };
        if (ph == 0) rows_at(0);

        const bool x_phase = ph != 1 && ph != 3;
        if (x_phase || (ph == 1 && !attends)) {
            const float *src = ph == 2 ? x1 : o - D;
            if constexpr (PARTS) {
                if (li && !(ph == 2 && attends)) small_add_parts(v, o - parts * D, parts, D, sums, a);
                if (ph == 2) small_add_parts(v, part1, a.heads, D, sums, a);
            } else if (ph == 2 || li) small_poll_x(v, src, D, a);
            lds_barrier();           // other waves still read xs and xraw
            const small_float_p w = ph == 4 ? (small_float_p)a.norm : ph == 2 ? small_norm(&l.ffn_norm) : ph == 0 ? small_norm(&l.attn_norm) : nullptr;
            small_stage_x(v, D, w, xraw, xs, red);
        }
        if (!x_phase) small_stage(ph == 1 ? o : ff, ph == 1 ? D : F, xs, a);

        g.run(xs, [&](uint32_t r, float up, float s) {
            if (ph == 0) {
                if (r < R) qs[r] = s;
                else if (r < 2 * R) knew[r - R] = float_to_half_bits(s);
                else vnew[r - 2 * R] = float_to_half_bits(s);
            } else if (ph == 4) {
                a.logits[r] = s;
                a.logits_host[r] = s;
            } else if (ph == 2) {
                const float f = up * s / (__expf(-s) + 1.f);
                if constexpr (PARTS) xraw[r] = f;          // the residual is in registers
                else small_publish(ff + r, f);
            }
            else small_publish((ph == 1 ? x1 : x2) + r, xraw[r] + s);
        });
        if (PARTS && ph == 2) {
            lds_barrier();
            if (nown) cols.publish(xraw, nown, own, D, part2 + blockIdx.x * D);
        }
        if (ph != 0) continue;

        lds_barrier();
        if (tid < R) {
            kc[(size_t)cur * D + tid] = knew[tid];
            vc[(size_t)cur * D + tid] = vnew[tid];
        }
        const float scale = rsqrtf((float)R);
        float qv[8], acc[8] = {}, den = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) qv[i] = qs[sub * 8 + i];
        for (uint32_t p0 = 0; p0 <= cur; p0 += BATCH * RPB) {
            if (p0) rows_at(p0);
#pragma unroll
            for (int j = 0; j < BATCH; j++) {
                const uint32_t p = p0 + j * RPB + rsel;
                uint4 kw4 = kr[j], vw4 = vr[j];
                if (p >= cur) {
                    kw4 = *reinterpret_cast<const uint4 *>(knew + sub * 8);
                    vw4 = *reinterpret_cast<const uint4 *>(vnew + sub * 8);
                }
                const uint32_t kw[4] = {kw4.x, kw4.y, kw4.z, kw4.w}, vw[4] = {vw4.x, vw4.y, vw4.z, vw4.w};
                const float ct[4] = {t0[j].x, t0[j].z, t1[j].x, t1[j].z}, st[4] = {t0[j].y, t0[j].w, t1[j].y, t1[j].w};
                float s = 0.f;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float kx = half_bits_to_float((uint16_t)(kw[i] & 0xffffu)), ky = half_bits_to_float((uint16_t)(kw[i] >> 16));
                    const float qx = qv[2 * i], qy = qv[2 * i + 1];
                    s = fmaf(ct[i], fmaf(qy, ky, qx * kx), s);
                    s = fmaf(st[i], fmaf(qx, ky, -(qy * kx)), s);
                }
                s = group_sum<LPR>(s);
                const bool in = p <= cur;
                const float e = in ? __expf(s * scale) : 0.f;
                den += sub == 0 ? e : 0.f;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    acc[2 * i] = fmaf(e, half_bits_to_float((uint16_t)(vw[i] & 0xffffu)), acc[2 * i]);
                    acc[2 * i + 1] = fmaf(e, half_bits_to_float((uint16_t)(vw[i] >> 16)), acc[2 * i + 1]);
                }
            }
        }
#pragma unroll
        for (int off = LPR; off < 64; off <<= 1) {
#pragma unroll
            for (int i = 0; i < 8; i++) acc[i] += __shfl_xor(acc[i], off, kWave);
            den += __shfl_xor(den, off, kWave);
        }
        if (lane < LPR) {
#pragma unroll
            for (int i = 0; i < 8; i++) part[wave][lane * 8 + i] = acc[i];
            if (lane == 0) part[wave][R] = den;
        }
        lds_barrier();
        if (tid < R) {
            float num = 0.f, all = 0.f;
#pragma unroll
            for (int w = 0; w < kSmallWaves; w++) {
                num += part[w][tid];
                all += part[w][R];
            }
            if constexpr (PARTS) xraw[tid] = num / all;
            else small_publish(o + blockIdx.x * R + tid, num / all);
        }
        if constexpr (PARTS) {
            lds_barrier();
            cols.publish(xraw, R / 32, R / 32, D, part1 + blockIdx.x * D);
        }
    }
}

}  // namespace lv
