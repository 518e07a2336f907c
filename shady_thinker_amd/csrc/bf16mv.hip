// bf16 matvec for the lm_head / tied embeddings: y[m, n] = sum_k bf16(W[n, k])
// * x[m, k], W row-major [N, K] (two bf16 per u32, low half first), x f32 or
// f16 [M, K], y f32 [M, N], M <= 8. Replaces src/shaders/bf16_matvec.wgsl:21-72
// (dispatched at src/model.rs:455-468, 824-831).
//
// A pure HBM stream (151936 x 2560 bf16 = 778 MB for one token of the tied embeddings).
// One token: one shift or mask and one f32 FMA per weight, far below the VALU
// rate, so no matrix cores (bf16mv_kernel):
//  * 8 lanes share a row: one 16-byte load per lane covers 128 contiguous
//    bytes of each of 8 rows per instruction (full cache lines), and a row's
//    8 partial sums meet in 3 cross-lane steps.
//  * x is staged once per workgroup in LDS as f32; the 8 lanes of a row read
//    different 32-byte pieces, which every row group shares (broadcast).
//  * Waves loop over row groups (8 rows) with kUnroll loads in flight per lane.
// Two to eight tokens: that kernel would be bound by its x reads (two 16-byte
// LDS reads per lane, token and 8 weights), so bf16mm_kernel takes them, on
// the matrix cores; see there.
#include "common.hpp"

#include <algorithm>

namespace {

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kThreads = 256;
constexpr int kUnroll = 8;  // 16-byte weight loads in flight per lane

template <bool F16X>
__global__ __launch_bounds__(kThreads) void bf16mv_kernel(const void *__restrict__ xp, const uint16_t *__restrict__ w,
                                                          float *__restrict__ y, int K, int N, int groups_per_wave) {
    extern __shared__ __align__(16) float xs[];  // [K]
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int r = lane >> 3;  // row within the group of 8
    const int c = lane & 7;   // 16-byte piece within a 128-byte row segment

    // x -> LDS (f32)
    for (int k = tid * 4; k < K; k += kThreads * 4) {  // K % 8 == 0
        f32x4 v;
        if constexpr (F16X) {
            const _Float16 *s = static_cast<const _Float16 *>(xp) + k;
            v = f32x4{(float)s[0], (float)s[1], (float)s[2], (float)s[3]};
        } else {
            v = *reinterpret_cast<const f32x4 *>(static_cast<const float *>(xp) + k);
        }
        *reinterpret_cast<f32x4 *>(&xs[k]) = v;
    }
    __syncthreads();

    const int nseg = K / 64;           // full 128-byte segments per row
    const int tail = (K % 64) / 8;     // 16-byte pieces in the last partial segment
    const int nsteps = nseg + (tail > 0 ? 1 : 0);
    const int ngroups = (N + 7) / 8;
    const int gw = blockIdx.x * (kThreads / 64) + wave;  // first group of this wave
    const int gstride = gridDim.x * (kThreads / 64);

    for (int gi = 0; gi < groups_per_wave; ++gi) {
        const int g = gw + gi * gstride;
        if (g >= ngroups) break;  // uniform per wave
        const int row = min(g * 8 + r, N - 1);
        const u32x4 *wr = reinterpret_cast<const u32x4 *>(w + (size_t)row * K);
        float acc = 0.0f;
        for (int s0 = 0; s0 < nsteps; s0 += kUnroll) {
            u32x4 wv[kUnroll];
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {
                // piece c of segment s; past the row's end: a clamped valid
                // address, masked below
                const int piece = min((s0 + u) * 8 + c, K / 8 - 1);
                wv[u] = __builtin_nontemporal_load(wr + piece);
            }
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {
                const int s = s0 + u;
                const bool ok = s < nseg || (s == nseg && c < tail);
                if (!ok) continue;
                const int k = (s * 8 + c) * 8;
                // bf16 -> f32 is the upper half of an f32: low half << 16,
                // high half masked (copied out of the vector first: a bit
                // cast straight from a vector element miscompiles)
                const unsigned w4[4] = {wv[u].x, wv[u].y, wv[u].z, wv[u].w};
                float wf[8];
#pragma unroll
                for (int h = 0; h < 4; ++h) {
                    const unsigned lo = w4[h] << 16, hi = w4[h] & 0xFFFF0000u;
                    wf[2 * h] = __builtin_bit_cast(float, lo);
                    wf[2 * h + 1] = __builtin_bit_cast(float, hi);
                }
                const f32x4 a = *reinterpret_cast<const f32x4 *>(&xs[k]);
                const f32x4 b = *reinterpret_cast<const f32x4 *>(&xs[k + 4]);
                acc = fmaf(wf[0], a.x, acc);
                acc = fmaf(wf[1], a.y, acc);
                acc = fmaf(wf[2], a.z, acc);
                acc = fmaf(wf[3], a.w, acc);
                acc = fmaf(wf[4], b.x, acc);
                acc = fmaf(wf[5], b.y, acc);
                acc = fmaf(wf[6], b.z, acc);
                acc = fmaf(wf[7], b.w, acc);
            }
        }
        // the row's 8 partial sums (lanes 8r .. 8r+7)
        acc += __shfl_xor(acc, 1);
        acc += __shfl_xor(acc, 2);
        acc += __shfl_xor(acc, 4);
        const int n = g * 8 + r;
        if (c == 0 && n < N) y[n] = acc;
    }
}

// ---------------------------------------------------------------- 2-8 tokens
// Exact products on v_mfma_f32_32x32x16_bf16: x (f32) is the sum of three
// bf16 values (its top 8 significant bits, the next 8, the last 8; f16 x: of
// two), and each product of two bf16 values is exact in f32. The first parts'
// products are summed over US segments at a time and those sums added in f32,
// the other parts' (2^-8 of them) have an accumulator of their own: one chain
// for all was 2.4 times further from 64 bits than the sums of the one-token
// kernel at 5120 x 264.
//  * Weights stay as they are and go HBM -> registers: lane (q, row, h) of a
//    load (q = lane / 32, row = lane / 4 % 8, h = lane % 4) takes 16-byte
//    piece 4 q + h of a 128-byte segment of its row, so a load covers whole
//    lines of 8 rows, four lanes side by side 64 bytes of one. In the MFMA
//    that makes 32 A rows (row, h) of two 8-k slots q; B column (m, h) holds
//    token m's x of pieces h and 4 + h. Of the 32 x 32 sums those with equal h
//    are the result (a quarter: 3 MFMAs of 32 cycles per KiB of weights are
//    still a quarter of the time those take to arrive), added over h at the
//    end of a row group.
//  * x is staged in LDS as f32 (16-byte chunk c of token m at c ^ f(m): no
//    bank conflicts) and split by each wave as it goes, in the shadow of the
//    loads (six bytes per x would not fit the LDS for every K taken here).
//  * Each wave keeps the next US segments of its row groups in flight while
//    it computes US.
//  * x is staged times 2^24 and the sums are taken times 2^-24: the last part
//    of the smallest f32 subnormal is then a normal bf16 value (2^-125), so
//    that no part of any x is lost, whatever the weights.
//  * A sum that is not finite (inf - inf or inf * 0 among the parts of an
//    infinite x or weight would make a NaN of an infinity; the scale overflows
//    from |x| = 2^104) is done again in plain f32, by the whole wave: a token
//    with a NaN or an infinity in it does so for every row.
// Bound by HBM. us with 2 / 4 / 5 / 8 tokens, the former kernel (a row's 8
// lanes reading every token's x, f32 FMAs; bound by those reads) and this one:
//   2560 x 151936  191 / 187 / 366 / 371   143-155 (5.0-5.4 TB/s)
//   4096 x 32000    68 /  71 / 183 / 189   50-53
//   1024 x 8192     10 /  10 /  15 /  16   7.9-8.2
// (One token: 130, 49.9 and 7.0 there, about 137, 52 and 8 here: it stays
// there.) Two row groups per wave at once, 2 or 8 segments per batch, or a
// contiguous run of groups per wave: within 3% at 151936 rows; two workgroups
// of 8 waves per CU: slower at 8192 rows (4096 x 8192 22 against 19).
constexpr int kMmWaves = 16;               // waves per workgroup at most, one workgroup per CU: 128 registers each
constexpr int US = 4;                      // segments (KiB of weights) per batch
constexpr int kRsrcWord3 = 0x00020000;     // raw 32-bit buffer data (gfx9-class)
constexpr unsigned kNoLoad = 0x80000000u;  // buffer offset past every resource: reads 0, touches no memory
constexpr int kNt = 2;                     // non-temporal loads: weights are read once
constexpr float kUp = 16777216.0f, kDown = 1.0f / kUp;  // x is staged times 2^24

__device__ __forceinline__ int x_swizzle(int m) { return (m & 1) | ((m & 2) << 2); }

template <int CTRL>
__device__ __forceinline__ float quad_add(float v) {
    return v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}

__device__ __forceinline__ unsigned top_halves(float a, float b) {  // bf16 of a (low) and b, cut off
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
__device__ __forceinline__ float cut(float v) { return __uint_as_float(__float_as_uint(v) & 0xFFFF0000u); }

template <bool F16X>
__global__ __launch_bounds__(64 * kMmWaves) void bf16mm_kernel(const void *__restrict__ xp, const uint16_t *__restrict__ w,
                                                               float *__restrict__ y, int M, int K, int N, int Kp) {
    extern __shared__ __align__(16) float xs[];  // [M][Kp], Kp = K up to a multiple of 64
    constexpr int NS = F16X ? 2 : 3;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane >> 5, mid = (lane >> 2) & 7, h = lane & 3;  // mid: weight row of A, token of B
    const int nsteps = Kp / 64, nb = (nsteps + US - 1) / US;
    const int ngroups = (N + 7) / 8, nwaves = gridDim.x * (blockDim.x >> 6);
    const int wid = blockIdx.x * (blockDim.x >> 6) + wave;
    // Batch b of row group g: its segments US b .. (past a row's end: the next
    // row's, against zeros of x; past the last row: nothing).
    const unsigned off0 = (unsigned)(mid * K * 2 + (4 * q + h) * 16);
    auto load = [&](u32x4 (&wv)[US], int g, int b) __attribute__((always_inline)) {
        const bool ok = g < ngroups;
        const int gj = ok ? g : 0;
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(w + (size_t)gj * 8 * K), (short)0, ok ? min(8, N - 8 * gj) * K * 2 : 0, kRsrcWord3);
#pragma unroll
        for (int u = 0; u < US; ++u) {
            unsigned o = US * b + u < nsteps ? off0 + (unsigned)(US * b + u) * 128u : kNoLoad;
            asm volatile("" : "+v"(o));  // (one load, not one on each side of a branch)
            wv[u] = __builtin_amdgcn_raw_buffer_load_b128(r, o, 0, kNt);
        }
    };
    const __amdgpu_buffer_rsrc_t rx =
        __builtin_amdgcn_make_buffer_rsrc((void *)xp, (short)0, M * K * (F16X ? 2 : 4), kRsrcWord3);
    // token m's x of k .. k + 3; past M or K zeros, by offset and not by a
    // branch: with one around each load and its store the loads of eight
    // tokens came one after the other (5120 x 264, 8 tokens of f16 x: 41 us)
    auto load_x = [&](int m, int k) __attribute__((always_inline)) {
        const unsigned o = m < M && k < K ? (unsigned)(m * K + k) * (F16X ? 2u : 4u) : kNoLoad;
        if constexpr (F16X) {
            const half4 s = __builtin_bit_cast(half4, __builtin_amdgcn_raw_buffer_load_b64(rx, o, 0, 0));
            return f32x4{(float)s[0], (float)s[1], (float)s[2], (float)s[3]};
        } else {
            return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, o, 0, 0));
        }
    };
    u32x4 wa[US], wb[US];
    load(wa, wid, 0);

    for (int c = tid; c < Kp / 4; c += blockDim.x) {
        f32x4 v[8];  // chunk c of every token, all loads in flight at once
#pragma unroll
        for (int m = 0; m < 8; ++m) v[m] = load_x(m, 4 * c);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < 8; ++m)
            if (m < M) *reinterpret_cast<f32x4 *>(&xs[m * Kp + 4 * (c ^ x_swizzle(m))]) = v[m] * kUp;
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

    const int mr = min(mid, M - 1);  // (columns past M repeat the last token and are not stored)
    const float *const xrow = xs + mr * Kp;
    const int sw = x_swizzle(mr), c0 = 2 * (4 * q + h);
    f32x16 acc, low;
    auto compute = [&](const u32x4 (&wv)[US], int b) __attribute__((always_inline)) {
        f32x16 top;
#pragma unroll
        for (int i = 0; i < 16; ++i) top[i] = 0.0f;
#pragma unroll
        for (int u = 0; u < US; ++u) {
            const int c = 16 * min(US * b + u, nsteps - 1) + c0;  // (past the end: weights are 0)
            const f32x4 lo4 = *reinterpret_cast<const f32x4 *>(xrow + 4 * (c ^ sw));
            const f32x4 hi4 = *reinterpret_cast<const f32x4 *>(xrow + 4 * ((c + 1) ^ sw));
            const float v[8] = {lo4.x, lo4.y, lo4.z, lo4.w, hi4.x, hi4.y, hi4.z, hi4.w};
            u32x4 p[NS];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float r0 = v[2 * e] - cut(v[2 * e]), r1 = v[2 * e + 1] - cut(v[2 * e + 1]);
                p[0][e] = top_halves(v[2 * e], v[2 * e + 1]);
                p[1][e] = top_halves(r0, r1);
                if constexpr (NS == 3) p[NS - 1][e] = top_halves(r0 - cut(r0), r1 - cut(r1));
            }
            const bf16x8 wf = __builtin_bit_cast(bf16x8, wv[u]);
            top = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf, __builtin_bit_cast(bf16x8, p[0]), top, 0, 0, 0);
#pragma unroll
            for (int s = 1; s < NS; ++s)
                low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf, __builtin_bit_cast(bf16x8, p[s]), low, 0, 0, 0);
        }
        acc += top;
    };
    auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = low[i] = 0.0f;
    };
    // Row n's sum for token m in plain f32, by all lanes.
    auto row_sum = [&](int n, int m) __attribute__((always_inline)) {
        const uint16_t *const wr = w + (size_t)n * K;
        float t = 0.0f;
#pragma unroll 1
        for (int k = 8 * lane; k < K; k += 512) {  // K % 8 == 0
            const u32x4 wv = *reinterpret_cast<const u32x4 *>(wr + k);
            f32x4 x2[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) x2[i] = load_x(m, k + 4 * i);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const unsigned we = wv[e >> 1];
                t = fmaf(__uint_as_float(e & 1 ? we & 0xFFFF0000u : we << 16), x2[e >> 2][e & 3], t);
            }
        }
#pragma unroll
        for (int d = 1; d < 64; d *= 2) t += __shfl_xor(t, d);
        return t;
    };
    auto store = [&](int g) __attribute__((always_inline)) {
        acc += low;
        // Lane: column l % 32 = (token, h), A rows 8 (i / 4) + 4 q + i % 4 =
        // (weight row 2 (i / 4) + q, h' = i % 4): its own h' = h, summed over
        // the quad; lane h keeps weight row 2 h + q.
        float out = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float a01 = h & 1 ? acc[4 * i + 1] : acc[4 * i], a23 = h & 1 ? acc[4 * i + 3] : acc[4 * i + 2];
            const float t = quad_add<0x4E>(quad_add<0xB1>(h & 2 ? a23 : a01));
            out = h == i ? t : out;
        }
        const int n = 8 * g + 2 * h + q;
        const bool mine = n < N && mid < M;
        const bool bad = mine && !(fabsf(out) <= 3.402823466e38f);
        out *= kDown;
        for (unsigned long long todo = __ballot(bad); todo; todo &= todo - 1) {
            const int l = __builtin_ctzll(todo);
            const float t = row_sum(8 * g + 2 * (l & 3) + (l >> 5), (l >> 2) & 7);  // lane l's row and token
            out = lane == l ? t : out;
        }
        if (mine) y[(size_t)mid * N + n] = out;
    };
    clear();
    int g = wid, b = 0;  // the batch in hand
    while (g < ngroups) {
        auto turn = [&](u32x4 (&cur)[US], u32x4 (&nxt)[US]) __attribute__((always_inline)) {
            const bool last = b + 1 == nb;
            const int gn = last ? g + nwaves : g, bn = last ? 0 : b + 1;
            load(nxt, gn, bn);
            __builtin_amdgcn_sched_barrier(0);
            compute(cur, b);
            if (last) {
                store(g);
                clear();
            }
            g = gn;
            b = bn;
        };
        turn(wa, wb);
        if (g >= ngroups) break;
        turn(wb, wa);
    }
}

template <bool F16X>
int launch_mv(st_context *ctx, const void *x, const uint16_t *w, float *y, int K, int N) {
    const int ngroups = (N + 7) / 8;
    const int waves_per_wg = kThreads / 64;
    // about 8 workgroups (32 waves) per CU, each wave a few row groups
    const int target_wgs = std::max(1, ctx->num_cus * 8);
    const int gpw = std::max(1, (ngroups + target_wgs * waves_per_wg - 1) / (target_wgs * waves_per_wg));
    const int wgs = (ngroups + gpw * waves_per_wg - 1) / (gpw * waves_per_wg);
    const size_t lds = (size_t)K * sizeof(float);
    auto kern = bf16mv_kernel<F16X>;
    if (lds > 64 * 1024)
        ST_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    st::launch(ctx, kern, dim3(wgs), dim3(kThreads), lds, x, w, y, K, N, gpw);
    return st::launch_check("bf16mv_kernel");
}

template <bool F16X>
int launch_mm(st_context *ctx, const void *x, const uint16_t *w, float *y, int M, int K, int N) {
    const int Kp = (K + 63) / 64 * 64, ngroups = (N + 7) / 8;
    const size_t lds = (size_t)M * Kp * sizeof(float);
    // One workgroup per CU, of up to 16 waves; few row groups: fewer waves.
    const int waves = std::min(kMmWaves, (ngroups + ctx->num_cus - 1) / ctx->num_cus);
    const int wgs = std::min(ctx->num_cus, (ngroups + waves - 1) / waves);
    auto kern = bf16mm_kernel<F16X>;
    if (lds > 64 * 1024)
        ST_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    st::launch(ctx, kern, dim3(wgs), dim3(64 * waves), lds, x, w, y, M, K, N, Kp);
    return st::launch_check("bf16mm_kernel");
}

template <bool F16X>
int by_m(st_context *ctx, const void *x, const uint16_t *w, float *y, int M, int K, int N) {
    return M == 1 ? launch_mv<F16X>(ctx, x, w, y, K, N) : launch_mm<F16X>(ctx, x, w, y, M, K, N);
}

}  // namespace

extern "C" int st_bf16_matvec(st_context *ctx, const void *x, int x_dtype, const uint16_t *w, float *y, int M, int K,
                              int N) {
    if (!ctx || !x || !w || !y) return st::fail(ST_ERR_INVALID, "st_bf16_matvec: NULL argument");
    if (M < 1 || M > 8) return st::fail(ST_ERR_SHAPE, "st_bf16_matvec: M=%d not in [1,8]", M);
    if (K <= 0 || K % 8 || N <= 0) return st::fail(ST_ERR_SHAPE, "st_bf16_matvec: K=%d (multiple of 8), N=%d", K, N);
    const int mt = M == 1 ? 1 : (M <= 4 ? 4 : 8);  // token rows of the LDS x copy
    if ((size_t)mt * K * sizeof(float) > 160 * 1024)
        return st::fail(ST_ERR_SHAPE, "st_bf16_matvec: M=%d K=%d too large for the LDS x copy", M, K);
    if (x_dtype != ST_F32 && x_dtype != ST_F16) return st::fail(ST_ERR_INVALID, "st_bf16_matvec: x_dtype %d", x_dtype);
    if (!st::aligned16(w) || !st::aligned16(x))
        return st::fail(ST_ERR_ALIGN, "st_bf16_matvec: x and w must be 16-byte aligned");
    return x_dtype == ST_F16 ? by_m<true>(ctx, x, w, y, M, K, N) : by_m<false>(ctx, x, w, y, M, K, N);
}
