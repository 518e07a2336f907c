// Skinny GPTQ int4 GEMM with x held in registers (gfx950): a few to a few
// dozen tokens against tiled weights (st_gptq_i4_repack),
//   y[m, n]  = sum_g s[g, n] * sum_{k in g} (q[k, n] - z[g, n]) * x[m, k]
// or silu(gate) * up of two such sums, x as f32, f16 or f32 silu(a) * b (f16: a
// pre-pass) (semantics of gptq_matvec.wgsl:51-58, fused_gate_up_silu_4t.wgsl:24-90 and
// fused_silu_gptq_4t.wgsl:26-81; the reference runs one token at a time).
//
//  * Exact products: (q - z) is an integer in [-16, 15], exact in f16 (the
//    f16 1024 bias: 1024 + q, minus 1024 + z). f16 x is used as is. f32 x
//    (and silu(a) * b) is scaled per token and wave by a power of two into
//    f16's range and split into hi + lo, two f16 values (about 22
//    significant bits): two MFMAs, into two accumulators. Each 64 or 128 k
//    sum into fresh f32 accumulators that are then added and scaled by s in f32.
//  * Work split. A workgroup owns a run of 16-column tiles, a K slice and a
//    block of tokens (16 f32 or 32 f16). Its waves split the slice's 128-k
//    units, U consecutive units each, and keep the MFMA A fragments of their
//    own units in registers (32 VGPRs per unit) for all the workgroup's
//    tiles: x is read, scaled and split once per workgroup, none of it is
//    shared through LDS, and no wave waits for another while weights stream.
//    Per tile each wave leaves its 16-column partial sums in LDS; after every
//    R / NSRC tiles the workgroup meets once and adds them in pairs (a fixed
//    order).
//  * Weights stream through a register ring of R tiles x U units per wave
//    (48-64 KiB in flight per CU); loads past the end use an out-of-range
//    buffer offset (no access), so every path issues the same loads.
//  * More tokens than a block: workgroups of the same tiles and other tokens
//    run side by side on one XCD, so the weights come from HBM once and from
//    that XCD's L2 after (on any XCDs, in grids that are no multiple of 8: 3
//    blocks 6% slower over 307 drawn prompts, up to 13%, 5 blocks 8%).
//  * Few tiles, or K beyond what the waves hold: K slices across workgroups,
//    f32 partials in the workspace, added in a fixed order by a reduce launch;
//    where those of all columns do not fit, the columns in several launches.
#pragma once
#include "common.hpp"
#include "i4frag.hpp"
#include "xcd.hpp"

#include <type_traits>

namespace st {
namespace xs {

using namespace i4;

constexpr int kTileN = 16;
constexpr int kMaxSplit = 16;              // K slices
constexpr int kRsrcWord3 = 0x00020000;     // raw 32-bit buffer data (gfx9-class)
constexpr int kNt = 2;                       // non-temporal loads: a workgroup reads its weights once
constexpr unsigned kNoLoad = 0x80000000u;  // buffer offset past every resource: reads 0, touches no memory

// X_F16G: f16 x against (q - z) s rounded once to f16 (the prefill GEMM's
// weights) instead of exact (q - z), s applied to the sums.
enum { X_F16 = 0, X_F32 = 1, X_F32_SILU = 2, X_F16G = 3 };

constexpr bool is_half(int xm) { return xm == X_F16 || xm == X_F16G; }  // one f16 value per x

constexpr int kWaves = 8;                   // waves per workgroup
// 128-k units per wave at most: their weights, fragments and sums are in
// registers, two f32 inputs of silu(a) * b at first too, and where they spill
// one unit less is faster or the same. us at 4 / 3 units: gate/up with zero
// points 4096 x 14336, 32 tokens, f32 x, group 128 36.8 / 31.8, group 256 38.5 /
// 33.4, f16 x 26.9 / 24.9 and 29.0 / 25.8. One source with zero points: 4 in
// groups 128 and 256 (f16 x: 8 registers spilled; f32 x, two units at a time,
// none; from 5% slower than 3 units, 3328 x 4096, to 5% faster, 4096 x 14336), 3
// in groups of 64 (20-28 spilled at 4: 4096 x 14336, f16 x, 23.1 / 16.6).
constexpr int max_units(int xm, int nsrc, int gs, bool hz) {
    return xm == X_F32_SILU ? 2 : xm == X_F16G || !hz ? 4 : gs == 64 || nsrc == 2 ? 3 : 4;
}
// Gate/up with zero points in groups of 64: three units spill 8-10 registers and
// take half as long again. Faster than two all the same where two need K slices
// for many columns (plan; 2560 x 12656, 31 tokens, 2 / 3 units 31.1 / 26.7 us,
// 2816 x 10160, 13 tokens, 16.4 / 19.7, 5632 x 9728 37.8 / 51.5).
constexpr bool spills(int xm, int nsrc, int gs, bool hz, int U) {
    return (xm == X_F32 || xm == X_F16) && nsrc == 2 && gs == 64 && hz && U == 3;
}
constexpr int block_tokens(int xm) { return is_half(xm) ? 32 : 16; }

struct Args {
    const void *x, *xb;  // [M, K]; xb: b of silu(a) * b
    const uint32_t *qw[2];
    const uint16_t *sc[2];
    const uint32_t *qz[2];
    void *y;
    float *part;  // K slices' partial sums (ks > 1)
    const float *rsc;  // or nullptr: factor of each token's y (one source)
    int zoff, M, K, N, tq, trem, uq, urem, ks, tblocks, f16out;  // tq, trem: tiles / runs; uq, urem: 128-k units / K slices
    int tile0, pn;  // the launch's first tile; columns of the partial sums
};

// launch_gs<XM, NSRC, GS> for the group size; groups: runs of tiles
template <int XM, int NSRC>
int launch(st_context *ctx, const Args &a, int gs, int groups, bool hz);

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

// The sum of p in pairs of pairs: a fixed order, each value rounded log2(n)
// times (in a row n - 1 times, at growing sums).
template <int n>
__device__ __forceinline__ float pair_sum(float (&p)[n]) {
    static_assert((n & (n - 1)) == 0, "a power of two");
#pragma unroll
    for (int d = 1; d < n; d *= 2)
#pragma unroll
        for (int i = 0; i < n; i += 2 * d) p[i] += p[i + d];
    return p[0];
}

template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}

// (x0, x1) * up -> hi = f16 pair, lo = f16 pair of what hi leaves (mixed
// precision FMAs: two instructions per pair of either).
__device__ __forceinline__ unsigned mix_hi(float x0, float x1, float up) {
    unsigned h;
    asm("v_fma_mixlo_f16 %0, %1, %3, 0 op_sel_hi:[0,0,0]\n\tv_fma_mixhi_f16 %0, %2, %3, 0 op_sel_hi:[0,0,0]"
        : "=&v"(h) : "v"(x0), "v"(x1), "v"(up));
    return h;
}
__device__ __forceinline__ unsigned mix_lo(float x0, float x1, float up, unsigned h) {
    unsigned l;
    asm("v_fma_mixlo_f16 %0, %1, %3, -%4 op_sel:[0,0,0] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %0, %2, %3, -%4 op_sel:[0,0,1] op_sel_hi:[0,0,1]"
        : "=&v"(l) : "v"(x0), "v"(x1), "v"(up), "v"(h));
    return l;
}

// XM: how x comes; NSRC: 1, or 2 (gate/up); U: 128-k units of a wave with
// the most (the others have one less); R: ring entries (one tile of one
// source each); HZ: zero points given (else z = 8).
template <int XM, int NSRC, int GS, int U, int R, bool HZ>
__global__ __launch_bounds__(64 * kWaves) void i4xs_kernel(Args a) {
    constexpr bool HALF = is_half(XM);  // one f16 value per x, two 16-row blocks
    constexpr bool ROUND = XM == X_F16G;
    constexpr bool SILU = XM == X_F32_SILU;
    constexpr bool SCALED = !HALF;  // x scaled by 2^(15 - ex) per token and wave
    constexpr int MB = HALF ? 2 : 1;      // 16-row blocks
    constexpr int TPB = 16 * MB;          // tokens per workgroup
    constexpr int NG = GS == 64 ? 2 : 1;  // groups per 128-k unit
    constexpr int EK = 4 / NG;            // MFMA steps (32 k) per group
    constexpr int RT = R / NSRC;          // tiles per round
    static_assert(R % NSRC == 0 && RT <= 4, "a round is whole tiles, their scales one load");
    // Per wave: the staging buffer of one unit's x (8 KB: 16 rows of f32 or
    // 32 of f16), later the wave's partial sums [R][MB][4][64] of a round.
    constexpr int WB = 8192;
    static_assert(R * MB * 1024 <= WB, "partial sums");
    __shared__ __align__(1024) unsigned char lds[kWaves * WB];
    __shared__ __align__(16) float down[kWaves][32];  // each wave's 2^(ex - 15) of its rows

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = lane >> 4, r16 = lane & 15;

    // XCD-major order: consecutive ids (first the token blocks of one tile
    // run, then its K slices) share an XCD, but for the 7 places where one
    // XCD's workgroups end.
    int id = xcd_order(blockIdx.x, gridDim.x);
    const int tok0 = (id % a.tblocks) * TPB;
    id /= a.tblocks;
    const int ksl = id % a.ks, grp = id / a.ks;
    // (the first ntiles % groups runs are one tile longer; likewise the K
    // slices' units, and the units of a slice over its waves)
    const int t0 = a.tile0 + grp * a.tq + min(grp, a.trem), nt = a.tq + (grp < a.trem ? 1 : 0);
    const int G = a.K / GS, K = a.K, N = a.N;
    const int us = a.uq + (ksl < a.urem ? 1 : 0);
    const int nu = us / kWaves + (wave < us % kWaves ? 1 : 0);  // this wave's units: U or U - 1 (less in short slices)
    const int ub = ksl * a.uq + min(ksl, a.urem) + wave * (us / kWaves) + min(wave, us % kWaves);

    // ------------------------------------------------------------- x loads
    // Lane (row l / 16, chunk l % 16) of load j takes 8 k of token row 4 j +
    // l / 16: whole rows of a unit per instruction. (The fragments' own
    // order, 16 rows side by side, would take four times the address
    // cycles.) Rows past M read nothing.
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)a.x, (short)0, 0x7FFFFFFF, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t rxb =
        __builtin_amdgcn_make_buffer_rsrc((void *)(SILU ? a.xb : a.x), (short)0, 0x7FFFFFFF, kRsrcWord3);
    constexpr int ES = HALF ? 2 : 4;  // bytes per x
    constexpr int XL = HALF ? 1 : 2;  // 16-byte loads per 8 k
    constexpr int XJ = TPB / 4;       // loads (of 4 rows) per unit
    u32x4 xr[U][XJ][XL], xbr[SILU ? U : 1][XJ][XL];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int j = 0; j < XJ; ++j) {
            const int t = tok0 + 4 * j + q;
            const bool ok = t < a.M && u < nu;
#pragma unroll
            for (int h = 0; h < XL; ++h) {
                const unsigned o = ok ? (unsigned)((t * K + (ub + u) * 128 + 8 * r16) * ES) + 16u * h : kNoLoad;
                xr[u][j][h] = __builtin_amdgcn_raw_buffer_load_b128(rx, o, 0, 0);
                if constexpr (SILU) xbr[u][j][h] = __builtin_amdgcn_raw_buffer_load_b128(rxb, o, 0, 0);
            }
        }
    __builtin_amdgcn_sched_barrier(0);

    // ---------------------------------------------------- weights, scales
    // Tiled words of group g: lane l's GS / 32 words at ((T G + g) 64 + l) GS / 32,
    // word 2 st + h = packed row GS / 8 g + 8 st + 2 (l / 16) + h.
    u32x4 ring[R][U];
    // Scales and zero words of a round: lane (q, r) loads those of column r
    // of the round's tile q, one load for all its tiles. The next round's
    // are loaded at a round's start, before the weights it requests, so
    // taking them over at its end waits for none of those.
    struct Meta {
        unsigned s[NSRC][U][NG], z[NSRC][U][NG];
    };
    Meta meta;
    const __amdgpu_buffer_rsrc_t rw0 = __builtin_amdgcn_make_buffer_rsrc((void *)a.qw[0], (short)0, 0x7FFFFFFF, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t rs0 = __builtin_amdgcn_make_buffer_rsrc((void *)a.sc[0], (short)0, 0x7FFFFFFF, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t rz0 = __builtin_amdgcn_make_buffer_rsrc((void *)(HZ ? (const void *)a.qz[0] : a.sc[0]),
                                                                         (short)0, 0x7FFFFFFF, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t rw1 = __builtin_amdgcn_make_buffer_rsrc((void *)a.qw[1], (short)0, 0x7FFFFFFF, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t rs1 = __builtin_amdgcn_make_buffer_rsrc((void *)a.sc[1], (short)0, 0x7FFFFFFF, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t rz1 = __builtin_amdgcn_make_buffer_rsrc((void *)(HZ ? (const void *)a.qz[1] : a.sc[1]),
                                                                         (short)0, 0x7FFFFFFF, kRsrcWord3);
    auto load_meta = [&](Meta &me, int t) __attribute__((always_inline)) {  // of the round starting at tile t
        const int n = min(kTileN * (t0 + t + q) + r16, N - 1);
        const bool mine = t + q < nt && q < RT;
#pragma unroll
        for (int src = 0; src < NSRC; ++src)
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const bool ok = mine && u < nu;
                const int uu = u < nu ? ub + u : 0;
#pragma unroll
                for (int j = 0; j < NG; ++j) {
                    const int g = GS == 64 ? 2 * uu + j : uu * 128 / GS;
                    me.s[src][u][j] =
                        __builtin_amdgcn_raw_buffer_load_b16(NSRC == 2 && src ? rs1 : rs0, ok ? (unsigned)n * 2u : kNoLoad, g * N * 2, 0);
                    if constexpr (HZ)
                        me.z[src][u][j] = __builtin_amdgcn_raw_buffer_load_b32(NSRC == 2 && src ? rz1 : rz0,
                                                                               ok ? (unsigned)(n >> 3) * 4u : kNoLoad, g * (N >> 3) * 4, 0);
                }
            }
    };
    auto load = [&](u32x4 (&it)[U], int src, int t) __attribute__((always_inline)) {
        const bool tok = t < nt;
        const int T = t0 + (tok ? t : 0);
        const __amdgpu_buffer_rsrc_t rw = NSRC == 2 && src ? rw1 : rw0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool ok = tok && u < nu;
            const int uu = ok ? ub + u : 0;  // (absent units: addresses in range, nothing read)
            // offsets pinned in VGPRs: left as selects on a uniform condition
            // the compiler makes two loads on two branches of each
            unsigned ow = ok ? (unsigned)(lane * (GS == 64 ? 8 : GS == 128 ? 16 : 32)) : kNoLoad;
            asm volatile("" : "+v"(ow));
            if constexpr (GS == 64) {
                const int so = (T * G + 2 * uu) * 512;
                const u32x2 w0 = __builtin_amdgcn_raw_buffer_load_b64(rw, ow, so, kNt);
                const u32x2 w1 = __builtin_amdgcn_raw_buffer_load_b64(rw, ow, so + 512, kNt);
                it[u] = u32x4{w0.x, w0.y, w1.x, w1.y};
            } else if constexpr (GS == 128) {
                it[u] = __builtin_amdgcn_raw_buffer_load_b128(rw, ow, (T * G + uu) * 1024, kNt);
            } else {
                it[u] = __builtin_amdgcn_raw_buffer_load_b128(rw, ow, (T * G + uu / 2) * 2048 + (uu & 1) * 16, kNt);
            }
        }
    };
    load_meta(meta, 0);
#pragma unroll
    for (int rr = 0; rr < R; ++rr) load(ring[rr], rr % NSRC, rr / NSRC);
    __builtin_amdgcn_sched_barrier(0);

    // ---------------------------------------------------------- x fragments
    // A fragments of v_mfma_f32_16x16x32_f16: lane (q, r) holds row r (token)
    // and the 8 k of word 2 st + h of lane block q: k = 64 st + 16 q + 8 h,
    // in the order of word_to_b.
    // xa[u][step][0..1]: hi and lo (f32), or the two row blocks (f16).
    // Each unit goes through the wave's own staging buffer (LDS accesses of a
    // wave complete in order, so nothing waits for other waves): 32 rows of
    // 256 bytes (tokens, or the hi and then the lo parts of 16), row r's
    // 16-byte chunk c at chunk c ^ r % 16: no bank conflicts on either side.
    half8 xa[U][4][2];
    unsigned char *const wl = lds + wave * WB;
    float up[XJ];  // the scale of this lane's row of each load
    if constexpr (SCALED) {
        // 2^ex just above the largest |x| of the wave's k of a token (its 16
        // lanes are one DPP row). Scaled, x lies below 2^15, so f16's
        // subnormal steps (2^-24) are 2^-39 of the largest value. (A NaN
        // leaves the maximum to the others and stays itself.)
#pragma unroll
        for (int j = 0; j < XJ; ++j) {
            if (tok0 + 4 * j >= a.M) continue;  // (uniform)
            float m = 0.f;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if constexpr (SILU) {  // the product replaces x's own registers
#pragma unroll
                    for (int h = 0; h < XL; ++h) {
                        f32x4 c = __builtin_bit_cast(f32x4, xr[u][j][h]);
                        const f32x4 d = __builtin_bit_cast(f32x4, xbr[u][j][h]);
#pragma unroll
                        for (int e = 0; e < 4; ++e) c[e] = silu_f(c[e]) * d[e];
                        xr[u][j][h] = __builtin_bit_cast(u32x4, c);
                    }
                }
                const f32x4 c0 = __builtin_bit_cast(f32x4, xr[u][j][0]);
                const f32x4 c1 = __builtin_bit_cast(f32x4, xr[u][j][XL - 1]);
                asm("v_max3_f32 %0, |%1|, |%2|, %0\n\tv_max3_f32 %0, |%3|, |%4|, %0"
                    : "+v"(m) : "v"(c0[0]), "v"(c0[1]), "v"(c0[2]), "v"(c0[3]));
                asm("v_max3_f32 %0, |%1|, |%2|, %0\n\tv_max3_f32 %0, |%3|, |%4|, %0"
                    : "+v"(m) : "v"(c1[0]), "v"(c1[1]), "v"(c1[2]), "v"(c1[3]));
            }
            // (an instruction of the compiler's own between the asm above and
            // the DPP moves: it keeps the wait states that a DPP read needs
            // after a VALU write only where it knows that write)
            m = __int_as_float(__float_as_int(m) & 0x7FFFFFFF);
            m = fmaxf(m, dpp_f<0xB1>(m));   // quad_perm [1,0,3,2]
            m = fmaxf(m, dpp_f<0x4E>(m));   // quad_perm [2,3,0,1]
            m = fmaxf(m, dpp_f<0x141>(m));  // row_half_mirror
            m = fmaxf(m, dpp_f<0x140>(m));  // row_mirror
            const int ex = max(__builtin_amdgcn_frexp_expf(m), -100);
            up[j] = __builtin_amdgcn_ldexpf(1.0f, 15 - ex);
            if (r16 == 0) down[wave][4 * j + q] = __builtin_amdgcn_ldexpf(1.0f, ex - 15);
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int j = 0; j < XJ; ++j) {
            if (tok0 + 4 * j >= a.M) continue;  // (uniform)
            const int row = 4 * j + q;
            unsigned char *const dst = wl + row * 256 + ((r16 ^ (row & 15)) << 4);
            if constexpr (!SCALED) {
                *reinterpret_cast<u32x4 *>(dst) = to_b_order(u < nu ? xr[u][j][0] : u32x4{0, 0, 0, 0});
            } else {
                const f32x4 c0 = __builtin_bit_cast(f32x4, xr[u][j][0]);
                const f32x4 c1 = __builtin_bit_cast(f32x4, xr[u][j][XL - 1]);
                u32x4 H, L;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    H[e] = mix_hi(c0[e], c1[e], up[j]);
                    L[e] = mix_lo(c0[e], c1[e], up[j], H[e]);
                }
                *reinterpret_cast<u32x4 *>(dst) = H;
                *reinterpret_cast<u32x4 *>(dst + 4096) = L;
            }
        }
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int s = 0; s < 4; ++s)
                xa[u][s][b] = *reinterpret_cast<const half8 *>(wl + 4096 * b + r16 * 256 + (((8 * (s >> 1) + 2 * q + (s & 1)) ^ r16) << 4));
    }
    f32x4 pw[MB];  // 2^(ex - 15) of the rows this lane's sums belong to (rows 4 q + i)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
        pw[mb] = SCALED ? *reinterpret_cast<const f32x4 *>(&down[wave][16 * mb + 4 * q]) : f32x4{1.f, 1.f, 1.f, 1.f};

    // ---------------------------------------------------------------- tiles
    float *const red = reinterpret_cast<float *>(lds);  // wave w's sums at w WB / 4
    // One ring entry's sums over NU units (U, or U - 1 in a wave with one unit
    // less). The units' MFMA chains are interleaved step by step: one chain
    // alone would leave the matrix pipe waiting for itself.
    auto entry = [&](auto NUC, auto RRC, int n7, f32x4 (&ys)[MB]) __attribute__((always_inline)) {
        constexpr int NU = decltype(NUC)::value, rr = decltype(RRC)::value, src = rr % NSRC;
        const int from = (r16 + 16 * (rr / NSRC)) * 4;  // the lane with this column's scale
        float sf[NU][NG];
        half2_t zlo[NU][NG], zhi[NU][NG];
#pragma unroll
        for (int u = 0; u < NU; ++u)
#pragma unroll
            for (int j = 0; j < NG; ++j) {
                const unsigned sw = (unsigned)__builtin_amdgcn_ds_bpermute(from, (int)meta.s[src][u][j]);
                sf[u][j] = (float)__builtin_bit_cast(_Float16, (uint16_t)sw);
                // f16 bits of 1024 + z (step 1) and -(64 + z) (step 1/16)
                unsigned z = 8u;
                if constexpr (HZ)
                    z = (((unsigned)__builtin_amdgcn_ds_bpermute(from, (int)meta.z[src][u][j]) >> (4 * n7)) & 0xF) + a.zoff;
                const unsigned zl = 0x6400u + z, zh = 0xD400u + 16u * z;
                zlo[u][j] = __builtin_bit_cast(half2_t, zl | (zl << 16));
                zhi[u][j] = __builtin_bit_cast(half2_t, zh | (zh << 16));
            }
        // [0..1]: the two row blocks, or (f32 x) the hi and the lo parts, whose
        // sums meet once per group: in one chain hi's sum, nearly exact by
        // itself, was rounded to lo's steps at every MFMA. Four units of them go
        // two by two: with all eight sums and zero points live six registers
        // spilled (3840 x 75936, 12 tokens, 45.6 / 40.0 us).
        constexpr int PU = SCALED && (NU == 4 || (NU == 3 && spills(XM, NSRC, GS, HZ, NU))) ? 2 : NU;  // units at a time
        constexpr int NA = ROUND ? (NU < 2 ? NU : 2) : PU;  // (ROUND: units may share accumulators)
        f32x4 acc[NA][2];
#pragma unroll
        for (int p = 0; p < NU; p += PU)
#pragma unroll
            for (int j = 0; j < NG; ++j) {
                if (!ROUND || j == 0)
#pragma unroll
                    for (int u = 0; u < NA; ++u) acc[u][0] = acc[u][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int e = 0; e < EK; ++e) {
                    const int step = EK * j + e;
                    half8 b[PU];
#pragma unroll
                    for (int u = 0; u < PU && p + u < NU; ++u) {
                        b[u] = word_to_b(ring[rr][p + u][step], zlo[p + u][j], zhi[p + u][j]);
                        if constexpr (ROUND) b[u] *= (_Float16)sf[p + u][j];  // (sf: an f16 value)
                    }
#pragma unroll
                    for (int u = 0; u < PU && p + u < NU; ++u)
                        acc[u % NA][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[p + u][step][0], b[u], acc[u % NA][0], 0, 0, 0);
#pragma unroll
                    for (int u = 0; u < PU && p + u < NU; ++u)
                        acc[u % NA][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[p + u][step][1], b[u], acc[u % NA][1], 0, 0, 0);
                }
                if constexpr (!ROUND)
#pragma unroll
                    for (int u = 0; u < PU && p + u < NU; ++u)
#pragma unroll
                        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                            for (int i = 0; i < 4; ++i)
                                ys[mb][i] = __builtin_fmaf(sf[p + u][j], SCALED ? acc[u][0][i] + acc[u][1][i] : acc[u][mb][i], ys[mb][i]);
            }
        if constexpr (ROUND)
#pragma unroll
            for (int u = 0; u < NA; ++u)
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) ys[mb] += acc[u][mb];
    };
    for (int t = 0; t < nt; t += RT) {
        Meta next;
        load_meta(next, t + RT);
        __builtin_amdgcn_sched_barrier(0);
        auto slot = [&](auto RRC) __attribute__((always_inline)) {
            constexpr int rr = decltype(RRC)::value, src = rr % NSRC;
            const int tt = t + rr / NSRC;
            f32x4 ys[MB];
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) ys[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
            const int n7 = (kTileN * (t0 + tt) + r16 < N ? r16 : N - 1) & 7;  // (column % 8: the nibble of its zero word)
            if (tt < nt) {  // (uniform)
                if (nu == U)
                    entry(std::integral_constant<int, U>{}, RRC, n7, ys);
                else if constexpr (U > 1)
                    entry(std::integral_constant<int, U - 1>{}, RRC, n7, ys);
            }
            load(ring[rr], src, tt + RT);
            __builtin_amdgcn_sched_barrier(0);
            if (rr == 0 && t > 0) lds_barrier();  // the last round's sums have been read
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    red[wave * (WB / 4) + ((rr * MB + mb) * 4 + i) * 64 + lane] = SCALED ? ys[mb][i] * pw[mb][i] : ys[mb][i];
        };
        slot(std::integral_constant<int, 0>{});
        slot(std::integral_constant<int, 1>{});
        if constexpr (R > 2) slot(std::integral_constant<int, 2>{});
        if constexpr (R > 3) slot(std::integral_constant<int, 3>{});
        meta = next;
        lds_barrier();
        constexpr int OUT = RT * MB * 256;  // sums of the round (per source)
        for (int o = threadIdx.x; o < OUT; o += 64 * kWaves) {
            const int l = o & 63, i = (o >> 6) & 3, mb = (o >> 8) % MB, rt = (o >> 8) / MB;
            float y[NSRC];
#pragma unroll
            for (int sr = 0; sr < NSRC; ++sr) {
                float p[kWaves];
#pragma unroll
                for (int w = 0; w < kWaves; ++w) p[w] = red[w * (WB / 4) + (((rt * NSRC + sr) * MB + mb) * 4 + i) * 64 + l];
                y[sr] = pair_sum(p);
            }
            const int m = tok0 + 16 * mb + 4 * (l >> 4) + i, nc = kTileN * (t0 + t + rt) + (l & 15);
            if (t + rt >= nt || m >= a.M || nc >= N) continue;
            if (a.ks > 1) {
#pragma unroll
                for (int sr = 0; sr < NSRC; ++sr) a.part[((size_t)(ksl * NSRC + sr) * a.M + m) * a.pn + nc - kTileN * a.tile0] = y[sr];
                continue;
            }
            const float yv = NSRC == 2 ? silu_f(y[0]) * y[NSRC - 1] : a.rsc ? y[0] * a.rsc[m] : y[0];
            if (a.f16out)
                static_cast<_Float16 *>(a.y)[(size_t)m * N + nc] = (_Float16)yv;
            else
                static_cast<float *>(a.y)[(size_t)m * N + nc] = yv;
        }
    }
}

template <int XM, int NSRC, int GS>
int launch_gs(st_context *ctx, const Args &a, int groups, bool hz) {
    const dim3 grid(groups * a.ks * a.tblocks), block(64 * kWaves);
    auto units = [&](auto UC, auto HZC) {
        constexpr int U = decltype(UC)::value;
        constexpr bool HZ = decltype(HZC)::value;
        if constexpr (U <= max_units(XM, NSRC, GS, HZ)) {
            st::launch(ctx, (i4xs_kernel<XM, NSRC, GS, U, U == 4 ? 2 : 4, HZ>), grid, block, 0, a);
            return st::launch_check("i4xs_kernel");
        } else
            return st::fail(ST_ERR_UNSUPPORTED, "i4xs: %d units per wave", U);
    };
    auto zeros = [&](auto UC) { return hz ? units(UC, std::true_type{}) : units(UC, std::false_type{}); };
    switch ((a.uq + (a.urem > 0) + kWaves - 1) / kWaves) {
        case 1: return zeros(std::integral_constant<int, 1>{});
        case 2: return zeros(std::integral_constant<int, 2>{});
        case 3: return zeros(std::integral_constant<int, 3>{});
        default: return zeros(std::integral_constant<int, 4>{});
    }
}

template <int XM, int NSRC>
int launch(st_context *ctx, const Args &a, int gs, int groups, bool hz) {
    switch (gs) {
        case 64: return launch_gs<XM, NSRC, 64>(ctx, a, groups, hz);
        case 128: return launch_gs<XM, NSRC, 128>(ctx, a, groups, hz);
        default: return launch_gs<XM, NSRC, 256>(ctx, a, groups, hz);
    }
}

}  // namespace xs
}  // namespace st
