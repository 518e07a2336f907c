// Host side of the skinny GPTQ kernel (i4xs.hpp): how a call is split over
// workgroups, the pre-passes (act-order gather, f16 silu(a) * b) and the
// reduction of K slices.
#include "i4xs.hpp"

#include <algorithm>

namespace st {
namespace xs {
// instantiated in i4xs_{f32,f32d,f32s,f16,f16d,f16g}.hip
extern template int launch<X_F32, 1>(st_context *, const Args &, int, int, bool);
extern template int launch<X_F32, 2>(st_context *, const Args &, int, int, bool);
extern template int launch<X_F32_SILU, 1>(st_context *, const Args &, int, int, bool);
extern template int launch<X_F16, 1>(st_context *, const Args &, int, int, bool);
extern template int launch<X_F16, 2>(st_context *, const Args &, int, int, bool);
extern template int launch<X_F16G, 1>(st_context *, const Args &, int, int, bool);
}  // namespace xs
}  // namespace st

namespace {

using namespace st::xs;

// y = epilogue(sum over slices s < ks of part[s][src]), the slices added in
// pairs (a fixed order), the epilogue silu(gate) * up for two sources. The
// partials are of pn columns from n0 on.
template <int NSRC, bool F16OUT>
__global__ __launch_bounds__(256) void i4xs_reduce_kernel(const float *__restrict__ part, void *__restrict__ y, int M,
                                                          int ks, const float *__restrict__ rsc, int N, int n0, int pn) {
    const int idx = blockIdx.x * 256 + threadIdx.x, MN = M * pn;
    if (idx >= MN) return;
    const int m = idx / pn;
    const size_t at = (size_t)m * N + n0 + (idx - m * pn);
    float t[NSRC][kMaxSplit];  // every slice's load issued before the first add
#pragma unroll
    for (int s = 0; s < kMaxSplit; ++s)
#pragma unroll
        for (int sr = 0; sr < NSRC; ++sr) t[sr][s] = s < ks ? part[(size_t)(s * NSRC + sr) * MN + idx] : 0.f;
    float v[NSRC];
#pragma unroll
    for (int sr = 0; sr < NSRC; ++sr) v[sr] = pair_sum(t[sr]);
    const float r = NSRC == 2 ? silu_f(v[0]) * v[NSRC - 1] : rsc ? v[0] * rsc[m] : v[0];
    if (F16OUT)
        static_cast<_Float16 *>(y)[at] = (_Float16)r;
    else
        static_cast<float *>(y)[at] = r;
}

// Act-order: xg[t, k] = x[t, perm[k]] (the sorted weight rows' order), or
// silu(x) * xb gathered so; four k per thread.
template <typename T, bool SILU>
__global__ __launch_bounds__(256) void i4xs_gather_kernel(const T *__restrict__ x, const T *__restrict__ xb,
                                                          const int32_t *__restrict__ perm, T *__restrict__ xg, int M, int K) {
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= (size_t)M * K) return;
    const size_t t = i / K, k = i % K;
    const int4 p = *reinterpret_cast<const int4 *>(perm + k);
    const int pk[4] = {p.x, p.y, p.z, p.w};
    const T *xr = x + t * K;
    T v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = xr[pk[e]];
    if constexpr (SILU) {
        const T *br = xb + t * K;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = silu_f(v[e]) * br[pk[e]];
    }
    __builtin_memcpy(xg + i, v, sizeof v);
}

// f16 silu(a) * b of a short prompt, once for all workgroups: row t's products
// (of k = perm[.] under act-order) times 2^-e rounded to f16, 2^e just above
// 2^-15 of the largest finite one, rsc[t] = 2^e. In the skinny kernel itself,
// which formed them before, every workgroup did so again for its K slice, and
// two inputs held its waves to two units (more slices). us per call, before /
// now: 77 tokens 9728 x 2560 29.1 / 26.4, 4096 x 2560 22.6 / 15.3; 160 tokens
// 11008 x 4096 51.9 / 43.6; with act-order (the GEMM before) 33 tokens 9728 x
// 2560 31.9 / 25.0. All of a row's loads are in flight at once: a block of 256
// threads in several passes took 8.0 us at 77 tokens, this 5.8.
constexpr int kSiluThreads = 1024;
__global__ __launch_bounds__(kSiluThreads) void i4xs_silu_kernel(const _Float16 *__restrict__ a, const _Float16 *__restrict__ b,
                                                                 const int32_t *__restrict__ perm, _Float16 *__restrict__ out,
                                                                 float *__restrict__ rsc, int K) {
    constexpr int P = 4;  // chunks of 8 k per thread: K <= 32768
    __shared__ float wmax[kSiluThreads / 64];
    const size_t base = (size_t)blockIdx.x * K;
    half8 g[P], u[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int k = (p * kSiluThreads + (int)threadIdx.x) * 8;
        g[p] = u[p] = half8{};
        if (k >= K) continue;
        if (perm) {
            const int4 p0 = *reinterpret_cast<const int4 *>(perm + k), p1 = *reinterpret_cast<const int4 *>(perm + k + 4);
            const int pk[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                g[p][e] = a[base + pk[e]];
                u[p][e] = b[base + pk[e]];
            }
        } else {
            g[p] = *reinterpret_cast<const half8 *>(a + base + k);
            u[p] = *reinterpret_cast<const half8 *>(b + base + k);
        }
    }
    float m = 0.f, h[P][8];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        if (p * kSiluThreads * 8 >= K) break;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            h[p][e] = silu_f((float)g[p][e]) * (float)u[p][e];
            m = fabsf(h[p][e]) <= 3.402823466e38f ? fmaxf(m, fabsf(h[p][e])) : m;
        }
    }
    for (int d = 32; d; d >>= 1) m = fmaxf(m, __shfl_xor(m, d));
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kSiluThreads / 64; ++w) m = fmaxf(m, wmax[w]);
    const int ex = max(__builtin_amdgcn_frexp_expf(m), -100) - 15;
    const float up = __builtin_amdgcn_ldexpf(1.0f, -ex);
    if (threadIdx.x == 0) rsc[blockIdx.x] = __builtin_amdgcn_ldexpf(1.0f, ex);
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int k = (p * kSiluThreads + (int)threadIdx.x) * 8;
        if (k >= K) break;
        half8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (_Float16)(h[p][e] * up);
        *reinterpret_cast<half8 *>(out + base + k) = o;
    }
}

struct Split {
    int ks = 0, groups = 0;  // ks = 0: no split fits
};

// K slices and tile runs: one workgroup per CU at most, the split with the
// least estimated time (us; MI355X, fitted to sweeps of both over the
// projections of 2560- and 4096-wide layers at 6-128 tokens): a wave's x
// costs x_us per unit, a tile tile_us per unit, and K slices a second launch
// plus their partial sums' way to memory and back.
Split plan(const st_context *ctx, int xm, int gs, bool hz, int M, int K, int N, int nsrc, size_t ws) {
    const int units = K / 128, ntiles = (N + kTileN - 1) / kTileN;
    const int tb = (M + block_tokens(xm) - 1) / block_tokens(xm);
    const bool half = is_half(xm);
    const int umax = max_units(xm, nsrc, gs, hz);
    const double x_us = half ? 0.4 : 0.8, tile_us = half ? 0.25 : 0.22;
    Split best;
    double least = 1e30;
    for (int ks = 1; ks <= std::min(kMaxSplit, units); ++ks) {
        const int U = ((units + ks - 1) / ks + kWaves - 1) / kWaves;
        if (U > umax) continue;
        const size_t bytes = ks > 1 ? (size_t)ks * nsrc * M * N * sizeof(float) : 0;
        if (bytes > ws) break;
        int groups = std::min(ntiles, std::max(1, ctx->num_cus / (ks * tb)));
        const int tq = (ntiles + groups - 1) / groups;
        const double waves = std::max(1.0, (double)groups * ks * tb / ctx->num_cus);  // (more token blocks than CUs)
        const double us = waves * U * (x_us + tile_us * nsrc * tq) * (spills(xm, nsrc, gs, hz, U) ? 1.55 : 1.0) +
                          (ks > 1 ? 1.7 + bytes * 2 / 3e6 : 0.0);
        if (us < least) {
            least = us;
            best.ks = ks;
            best.groups = groups;
        }
    }
    return best;
}

// The act-order gather and the f16 silu(a) * b pre-pass write to the workspace
// (x, then the rows' scales); false: it holds too little.
bool pre_pass(const st_context *ctx, const st::XsCall &c, size_t *off, size_t *rsc_off) {
    const bool half = c.x_f16, silu = c.xb != nullptr;
    *off = *rsc_off = 0;
    if (!c.perm && !(half && silu)) return true;
    *rsc_off = *off = ((size_t)c.M * c.K * (half ? 2 : 4) + 255) & ~size_t(255);
    if (half && silu) *off = (*off + (size_t)c.M * sizeof(float) + 255) & ~size_t(255);
    return ctx->ws && *off <= ctx->ws_bytes;
}

}  // namespace

namespace st {

int int4_xs(st_context *ctx, const XsCall &c) {
    const bool half = c.x_f16, silu = c.xb != nullptr;
    // (f16 silu(a) * b: exact weights, so that only the product is rounded)
    int xm = half ? (c.round_w && !silu ? X_F16G : X_F16) : (silu ? X_F32_SILU : X_F32);
    // act-order, and f16 silu(x) * xb: x (or the product) goes to the workspace first
    const bool pre = c.perm || (half && silu);
    size_t off, rsc_off;
    if (!pre_pass(ctx, c, &off, &rsc_off)) return -1;
    if (pre && silu && !half) xm = X_F32;
    const bool hz = c.qz[0] != nullptr;
    const int ntiles = (c.N + kTileN - 1) / kTileN;
    const size_t left = ctx->ws ? ctx->ws_bytes - off : 0;
    auto plan_tiles = [&](int tiles) { return plan(ctx, xm, c.gs, hz, c.M, c.K, std::min(tiles * kTileN, c.N), c.nsrc, left); };
    // Partial sums of all columns that do not fit: half the columns per launch,
    // a quarter, ..., at least a tile per CU. (8 MiB of workspace, an lm_head of 4608
    // x 152064, 9 / 32 tokens: 93 / 229 us, on the integer-limb kernels 186 / 463.)
    int run = ntiles;  // tiles per launch
    Split sp = plan_tiles(run);
    while (!sp.ks && c.parts && run >= 2 * ctx->num_cus) sp = plan_tiles(run = (run + 1) / 2);
    if (!sp.ks) return -1;
    Args a{};
    a.x = c.x;
    a.xb = c.xb;
    if (pre) {
        a.x = ctx->ws;
        a.xb = nullptr;
        if (half && silu) a.rsc = reinterpret_cast<float *>(reinterpret_cast<char *>(ctx->ws) + rsc_off);
    }
    if (pre && !c.gathered) {
        void *xg = ctx->ws;
        const dim3 g((unsigned)(((size_t)c.M * c.K / 4 + 255) / 256)), b(256);
        if (half && silu)
            st::launch(ctx, i4xs_silu_kernel, dim3(c.M), dim3(kSiluThreads), 0, static_cast<const _Float16 *>(c.x),
                       static_cast<const _Float16 *>(c.xb), c.perm, static_cast<_Float16 *>(xg),
                       reinterpret_cast<float *>(reinterpret_cast<char *>(ctx->ws) + rsc_off), c.K);
        else if (half)
            st::launch(ctx, i4xs_gather_kernel<uint16_t, false>, g, b, 0, static_cast<const uint16_t *>(c.x),
                       static_cast<const uint16_t *>(nullptr), c.perm, static_cast<uint16_t *>(xg), c.M, c.K);
        else if (silu)
            st::launch(ctx, i4xs_gather_kernel<float, true>, g, b, 0, static_cast<const float *>(c.x),
                       static_cast<const float *>(c.xb), c.perm, static_cast<float *>(xg), c.M, c.K);
        else
            st::launch(ctx, i4xs_gather_kernel<float, false>, g, b, 0, static_cast<const float *>(c.x),
                       static_cast<const float *>(nullptr), c.perm, static_cast<float *>(xg), c.M, c.K);
        if (int rc = launch_check(half && silu ? "i4xs_silu_kernel" : "i4xs_gather_kernel")) return rc;
    }
    for (int i = 0; i < 2; ++i) {
        const int j = i < c.nsrc ? i : 0;
        a.qw[i] = c.qw[j];
        a.sc[i] = c.sc[j];
        a.qz[i] = c.qz[j];
    }
    const int units = c.K / 128;
    a.y = c.y;
    a.zoff = c.zoff;
    a.M = c.M;
    a.K = c.K;
    a.N = c.N;
    a.tblocks = (c.M + block_tokens(xm) - 1) / block_tokens(xm);
    a.f16out = c.y_f16;
    for (a.tile0 = 0; a.tile0 < ntiles; a.tile0 += run) {
        const int tiles = std::min(run, ntiles - a.tile0);
        if (tiles < run) sp = plan_tiles(tiles);  // (the last launch's, which fits where `run` tiles do)
        a.pn = std::min(tiles * kTileN, c.N - a.tile0 * kTileN);
        a.part = sp.ks > 1 ? reinterpret_cast<float *>(reinterpret_cast<char *>(ctx->ws) + off) : nullptr;
        a.tq = tiles / sp.groups;
        a.trem = tiles % sp.groups;
        a.uq = units / sp.ks;
        a.urem = units % sp.ks;
        a.ks = sp.ks;
        int rc;
        switch (xm) {
            case X_F32: rc = c.nsrc == 2 ? xs::launch<X_F32, 2>(ctx, a, c.gs, sp.groups, hz) : xs::launch<X_F32, 1>(ctx, a, c.gs, sp.groups, hz); break;
            case X_F16: rc = c.nsrc == 2 ? xs::launch<X_F16, 2>(ctx, a, c.gs, sp.groups, hz) : xs::launch<X_F16, 1>(ctx, a, c.gs, sp.groups, hz); break;
            case X_F16G: rc = xs::launch<X_F16G, 1>(ctx, a, c.gs, sp.groups, hz); break;
            default: rc = xs::launch<X_F32_SILU, 1>(ctx, a, c.gs, sp.groups, hz); break;
        }
        if (rc) return rc;
        if (sp.ks == 1) continue;
        const dim3 g((c.M * a.pn + 255) / 256), b(256);
        const int n0 = a.tile0 * kTileN;
        if (c.nsrc == 2)
            c.y_f16 ? st::launch(ctx, i4xs_reduce_kernel<2, true>, g, b, 0, a.part, a.y, c.M, sp.ks, a.rsc, c.N, n0, a.pn)
                    : st::launch(ctx, i4xs_reduce_kernel<2, false>, g, b, 0, a.part, a.y, c.M, sp.ks, a.rsc, c.N, n0, a.pn);
        else
            c.y_f16 ? st::launch(ctx, i4xs_reduce_kernel<1, true>, g, b, 0, a.part, a.y, c.M, sp.ks, a.rsc, c.N, n0, a.pn)
                    : st::launch(ctx, i4xs_reduce_kernel<1, false>, g, b, 0, a.part, a.y, c.M, sp.ks, a.rsc, c.N, n0, a.pn);
        if (int rr = launch_check("i4xs_reduce_kernel")) return rr;
    }
    return ST_OK;
}

// Fitted to 1800 drawn calls of 33-256 tokens (MI355X, cold weights: within 6% rms).
double int4_xs_us(const st_context *ctx, const XsCall &c, double *pre_us) {
    const double MK = (double)c.M * c.K, MN = (double)c.M * c.N;
    const bool silu = c.xb != nullptr;
    *pre_us = (c.perm ? 3.4e-6 * MK + (silu ? 0.0 : 2.1) : 0.0) + (silu ? 3.8 + 1.7e-6 * MK : 0.0);
    size_t off, rsc_off;
    if (!pre_pass(ctx, c, &off, &rsc_off)) return 1e30;
    const int xm = silu ? X_F16 : X_F16G, tb = (c.M + block_tokens(xm) - 1) / block_tokens(xm);
    const Split sp = plan(ctx, xm, c.gs, silu && c.qz[0], c.M, c.K, c.N, 1, ctx->ws ? ctx->ws_bytes - off : 0);
    if (!sp.ks) return 1e30;
    const int U = ((c.K / 128 + sp.ks - 1) / sp.ks + kWaves - 1) / kWaves;
    const int tq = ((c.N + kTileN - 1) / kTileN + sp.groups - 1) / sp.groups;
    const double waves = std::max(1.0, (double)sp.groups * sp.ks * tb / ctx->num_cus);
    const double us = 4.0 + 1.0e-6 * (MK + MN) + waves * U * (0.93 + (c.gs == 64 ? 0.40 : 0.35) * tq);
    return us + (sp.ks > 1 ? 2.4 + 1.4e-6 * sp.ks * MN : 0.0);
}

}  // namespace st
