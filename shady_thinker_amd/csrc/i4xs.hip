// Host side of the skinny GPTQ kernel (i4xs.hpp): how a call is split over
// workgroups, the act-order gather and the reduction of K slices.
#include "i4xs.hpp"

#include <algorithm>

namespace st {
namespace xs {
// instantiated in i4xs_{f32,f32d,f32s,f16,f16d,f16s,f16g}.hip
extern template int launch<X_F32, 1>(st_context *, const Args &, int, int, bool);
extern template int launch<X_F32, 2>(st_context *, const Args &, int, int, bool);
extern template int launch<X_F32_SILU, 1>(st_context *, const Args &, int, int, bool);
extern template int launch<X_F16, 1>(st_context *, const Args &, int, int, bool);
extern template int launch<X_F16, 2>(st_context *, const Args &, int, int, bool);
extern template int launch<X_F16G, 1>(st_context *, const Args &, int, int, bool);
extern template int launch<X_F16_SILU, 1>(st_context *, const Args &, int, int, bool);
}  // namespace xs
}  // namespace st

namespace {

using namespace st::xs;

// y = epilogue(sum over slices s < ks of part[s][src]), the slices added in
// order (deterministic), the epilogue silu(gate) * up for two sources.
template <int NSRC, bool F16OUT>
__global__ __launch_bounds__(256) void i4xs_reduce_kernel(const float *__restrict__ part, void *__restrict__ y, int MN,
                                                          int ks) {
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= MN) return;
    float t[kMaxSplit][NSRC];  // every slice's load issued before the first add
#pragma unroll
    for (int s = 0; s < kMaxSplit; ++s)
#pragma unroll
        for (int sr = 0; sr < NSRC; ++sr) t[s][sr] = s < ks ? part[(size_t)(s * NSRC + sr) * MN + idx] : 0.f;
    float v[NSRC];
#pragma unroll
    for (int sr = 0; sr < NSRC; ++sr) {
        v[sr] = 0.f;
#pragma unroll
        for (int s = 0; s < kMaxSplit; ++s)
            if (s < ks) v[sr] += t[s][sr];
    }
    const float r = NSRC == 2 ? silu_f(v[0]) * v[NSRC - 1] : v[0];
    if (F16OUT)
        static_cast<_Float16 *>(y)[idx] = (_Float16)r;
    else
        static_cast<float *>(y)[idx] = r;
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

struct Split {
    int ks = 0, groups = 0;  // ks = 0: no split fits
};

// K slices and tile runs: one workgroup per CU at most, the split with the
// least estimated time (us; MI355X, fitted to sweeps of both over the
// projections of 2560- and 4096-wide layers at 6-128 tokens): a wave's x
// costs x_us per unit, a tile tile_us per unit, and K slices a second launch
// plus their partial sums' way to memory and back.
Split plan(const st_context *ctx, int xm, int M, int K, int N, int nsrc, size_t ws) {
    const int units = K / 128, ntiles = (N + kTileN - 1) / kTileN;
    const int tb = (M + block_tokens(xm) - 1) / block_tokens(xm);
    const bool half = is_half(xm), silu = xm == X_F32_SILU || xm == X_F16_SILU;
    const int umax = silu ? 2 : kMaxUnits;
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
        const double us = waves * U * (x_us + tile_us * nsrc * tq) + (ks > 1 ? 1.7 + bytes * 2 / 3e6 : 0.0);
        if (us < least) {
            least = us;
            best.ks = ks;
            best.groups = groups;
        }
    }
    return best;
}

}  // namespace

namespace st {

int int4_xs(st_context *ctx, const XsCall &c) {
    const bool half = c.x_f16, silu = c.xb != nullptr;
    int xm = half ? (silu ? X_F16_SILU : c.round_w ? X_F16G : X_F16) : (silu ? X_F32_SILU : X_F32);
    // act-order: x (or silu(x) * xb, f32 only) gathered into the workspace first
    size_t off = 0;
    if (c.perm) {
        if (half && silu) return -1;
        off = ((size_t)c.M * c.K * (half ? 2 : 4) + 255) & ~size_t(255);
        if (!ctx->ws || off > ctx->ws_bytes) return -1;
        if (silu) xm = X_F32;
    }
    const Split sp = plan(ctx, xm, c.M, c.K, c.N, c.nsrc, ctx->ws ? ctx->ws_bytes - off : 0);
    if (!sp.ks) return -1;
    Args a{};
    a.x = c.x;
    a.xb = c.xb;
    if (c.perm) {
        void *xg = ctx->ws;
        const dim3 g((unsigned)(((size_t)c.M * c.K / 4 + 255) / 256)), b(256);
        if (half)
            st::launch(ctx, i4xs_gather_kernel<uint16_t, false>, g, b, 0, static_cast<const uint16_t *>(c.x),
                       static_cast<const uint16_t *>(nullptr), c.perm, static_cast<uint16_t *>(xg), c.M, c.K);
        else if (silu)
            st::launch(ctx, i4xs_gather_kernel<float, true>, g, b, 0, static_cast<const float *>(c.x),
                       static_cast<const float *>(c.xb), c.perm, static_cast<float *>(xg), c.M, c.K);
        else
            st::launch(ctx, i4xs_gather_kernel<float, false>, g, b, 0, static_cast<const float *>(c.x),
                       static_cast<const float *>(nullptr), c.perm, static_cast<float *>(xg), c.M, c.K);
        if (int rc = launch_check("i4xs_gather_kernel")) return rc;
        a.x = xg;
        a.xb = nullptr;
    }
    for (int i = 0; i < 2; ++i) {
        const int j = i < c.nsrc ? i : 0;
        a.qw[i] = c.qw[j];
        a.sc[i] = c.sc[j];
        a.qz[i] = c.qz[j];
    }
    const bool hz = c.qz[0] != nullptr;
    const int units = c.K / 128, ntiles = (c.N + kTileN - 1) / kTileN;
    a.y = c.y;
    a.part = sp.ks > 1 ? reinterpret_cast<float *>(reinterpret_cast<char *>(ctx->ws) + off) : nullptr;
    a.zoff = c.zoff;
    a.M = c.M;
    a.K = c.K;
    a.N = c.N;
    a.tq = ntiles / sp.groups;
    a.trem = ntiles % sp.groups;
    a.uq = units / sp.ks;
    a.urem = units % sp.ks;
    a.ks = sp.ks;
    a.tblocks = (c.M + block_tokens(xm) - 1) / block_tokens(xm);
    a.f16out = c.y_f16;
    int rc;
    switch (xm) {
        case X_F32: rc = c.nsrc == 2 ? xs::launch<X_F32, 2>(ctx, a, c.gs, sp.groups, hz) : xs::launch<X_F32, 1>(ctx, a, c.gs, sp.groups, hz); break;
        case X_F16: rc = c.nsrc == 2 ? xs::launch<X_F16, 2>(ctx, a, c.gs, sp.groups, hz) : xs::launch<X_F16, 1>(ctx, a, c.gs, sp.groups, hz); break;
        case X_F16G: rc = xs::launch<X_F16G, 1>(ctx, a, c.gs, sp.groups, hz); break;
        case X_F32_SILU: rc = xs::launch<X_F32_SILU, 1>(ctx, a, c.gs, sp.groups, hz); break;
        default: rc = xs::launch<X_F16_SILU, 1>(ctx, a, c.gs, sp.groups, hz); break;
    }
    if (rc || sp.ks == 1) return rc;
    const int mn = c.M * c.N;
    const dim3 g((mn + 255) / 256), b(256);
    if (c.nsrc == 2)
        c.y_f16 ? st::launch(ctx, i4xs_reduce_kernel<2, true>, g, b, 0, a.part, a.y, mn, sp.ks)
                : st::launch(ctx, i4xs_reduce_kernel<2, false>, g, b, 0, a.part, a.y, mn, sp.ks);
    else
        c.y_f16 ? st::launch(ctx, i4xs_reduce_kernel<1, true>, g, b, 0, a.part, a.y, mn, sp.ks)
                : st::launch(ctx, i4xs_reduce_kernel<1, false>, g, b, 0, a.part, a.y, mn, sp.ks);
    return launch_check("i4xs_reduce_kernel");
}

}  // namespace st
