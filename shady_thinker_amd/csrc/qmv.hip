// C entry points of the decode kernels (GPTQ int4 and INT8 matvec / skinny
// GEMM) and the upload-time GPTQ repack. The kernel itself is in
// qmv_kernel.hpp; see there for the design.
#include "qmv_kernel.hpp"

namespace st {
namespace qmv {
// defined in qmv_i4_p{0,1}.hip, qmv_i4t_p{0,1}.hip, qmv_i8.hip
template <>
int dispatch<FMT_I4, false>(st_context *, Params &, int, int);
template <>
int dispatch<FMT_I4, true>(st_context *, Params &, int, int);
template <>
int dispatch<FMT_I4T, false>(st_context *, Params &, int, int);
template <>
int dispatch<FMT_I4T, true>(st_context *, Params &, int, int);
template <>
int dispatch<FMT_I8, false>(st_context *, Params &, int, int);
template <>
int dispatch<FMT_I8T, false>(st_context *, Params &, int, int);
}  // namespace qmv
}  // namespace st

namespace {

using namespace st::qmv;
using QmvParams = st::qmv::Params;

// Re-tile GPTQ qweight [K/8, N]: tile T (16 columns), group g becomes 64
// lanes x (gs/32) words, lane (q, c) holding, for each 64-k step st and h in
// {0, 1}, word [g*gs/8 + 8 st + 2q + h][16T + c]. Values are unchanged.
__global__ __launch_bounds__(256) void repack_kernel(const uint32_t *__restrict__ qw, uint32_t *__restrict__ out, int K,
                                                     int N, int gs, int ntiles) {
    const int wpl = gs / 32;  // words per lane per group
    const long long total = (long long)ntiles * (K / gs) * 64 * wpl;
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= total) return;
    const int j = (int)(idx % wpl);
    const int lane = (int)((idx / wpl) % 64);
    const long long tg = idx / ((long long)wpl * 64);
    const int g = (int)(tg % (K / gs));
    const int T = (int)(tg / (K / gs));
    const int q = lane >> 4, c = lane & 15;
    const int st = j >> 1, h = j & 1;
    const int n = min(16 * T + c, N - 1);
    const size_t pr = (size_t)g * (gs / 8) + st * 8 + 2 * q + h;
    out[idx] = qw[pr * N + n];
}

// Re-tile INT8 w [N, K]: tile T (16 rows), group u (128 k), lane (q, c)
// gets 32 contiguous bytes, k = 128 u + 16 q + 64 st + j (st < 2, j < 16) of
// row 16 T + c (rows past N repeat row N - 1). One thread per 16 bytes.
__global__ __launch_bounds__(256) void repack8_kernel(const int8_t *__restrict__ w, int8_t *__restrict__ out, int K,
                                                      int N, int ntiles) {
    const int units = K / 128;
    const long long total = (long long)ntiles * units * 64 * 2;
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= total) return;
    const int st = (int)(idx & 1);
    const int lane = (int)((idx >> 1) & 63);
    const long long tu = idx >> 7;
    const int u = (int)(tu % units);
    const int T = (int)(tu / units);
    const int n = min(16 * T + (lane & 15), N - 1);
    const size_t k0 = (size_t)u * 128 + 16 * (lane >> 4) + 64 * st;
    reinterpret_cast<uint4 *>(out)[idx] = *reinterpret_cast<const uint4 *>(w + (size_t)n * K + k0);
}

// The GPTQ entry points take an f16-MFMA kernel (tiled weights, with or
// without act-order) from a few tokens on. Times (us per call in a graph, cold
// weights, MI355X; integer-limb kernels against i4xs.hpp):
//   narrow linears (at most one 16-column tile per CU)
//     4096 x 4096           4 tokens  6.3 /  7.7   8 tokens  8.8 /  7.7
//     11008 x 4096                   10.6 / 11.6             13.6 / 12.1
//     silu(a) b, 4096 x 4096          8.4 /  9.3              9.9 /  9.6
//     act-order 4096 x 4096          14.4 /  9.7             13.1 /  9.9
//   wide: 2560 x 151936     4 tokens 39   / 42     5 tokens 77   / 42
// so from 5 tokens on; narrow linears with K below 2048 keep the limb kernels to
// 8 tokens. Under act-order the limb kernels gather x in every workgroup, which
// 3 and 4 tokens of a long x make dearer than the skinny kernel's gather launch
// (narrow linears drawn, limb / skinny: 3 tokens, K 1024-2600 0.86, to 4200 0.91,
// above 1.17; 4 tokens 0.92, 1.05, 1.31): there from M K = 3 x 4096, silu(a) b
// from 3 tokens (1.1-4.1).
constexpr int kF16MinM = 5;
constexpr int kF16MinMActOrder = 3;
constexpr int kF16MinMKActOrder = 3 * 4096;
constexpr int kF16MinMShortK = 9;
constexpr int kF16ShortK = 2048;

// Wide linears whose tokens fill 16 MFMA rows or less (8 tokens of f32 x, 16 of
// f16): i4mm.hip for gate/up (8 tokens of f32 x, i4mm / i4xs: 2560 x 9728 9.8 /
// 11.8 us, 4096 x 11008 13.6 / 14.5) and for one source by its tiles per CU (i4mm
// time over i4xs's, 400 drawn calls of 5-16 tokens, f32 x / f16 x):
//   below 3    2560 x 10240 7.5 / 8.4 us; but in groups of 64 with f32 x and at
//              most 2, where i4mm's 8-byte weight loads hold too little in
//              flight, i4xs (6 tokens: 4096 x 8000 12.0 / 10.2, 8192 x 6144
//              19.8 / 12.4; 4096 x 10240, 2.5 per CU, 10.5 / 11.6)
//   3 to 4     1.06 / 1.04 (in groups of 256 0.94 / 0.97): i4xs
//   4 to 6     0.93 / 0.87
//   6 to 8     0.98 / 0.88
//   above      1.30 / 1.15: more tiles than i4mm's workgroups take at once
// From 9 tokens of f32 x and 17 of f16 on i4xs is the faster one of the two in
// most shapes, not in all (f16 x of 17-32 tokens on 2-8 tiles per CU: 40 of 226
// drawn calls ran 4-30% faster on a two-row-block i4mm, which is gone).
bool use_i4mm(const st_context *ctx, const QmvParams &p, int ntiles, int nsrc, int xm) {
    const int ncu = ctx->num_cus;
    if (xm == XM_SILU || ntiles <= ncu || p.M > (xm == XM_F32 ? 8 : 16)) return false;
    if (nsrc == 2) return true;
    if (ntiles < 3 * ncu) return !(xm == XM_F32 && p.gs == 64 && ntiles <= 2 * ncu);
    return ntiles > 4 * ncu && ntiles <= (xm == XM_F32 ? 6 : 8) * ncu;
}

// -1: not taken.
int launch_f16(st_context *ctx, const QmvParams &p, bool tiled, int nsrc, int xm) {
    const int ntiles = (p.N + kTileN - 1) / kTileN;
    const bool few = ntiles <= ctx->num_cus;
    int dflt = kF16MinM;
    if (few && !p.perm && p.K < kF16ShortK) dflt = kF16MinMShortK;
    if (few && p.perm && (xm == XM_SILU || (long long)p.M * p.K >= kF16MinMKActOrder)) dflt = kF16MinMActOrder;
    const int min_m = std::max(2, st::tune(ctx, ST_TUNE_I4MM_MIN_M, dflt));
    const int min_tiles = st::tune(ctx, ST_TUNE_I4MM_MIN_TILES, ctx->num_cus + 1);
    const bool split = few && st::tune(ctx, ST_TUNE_I4MM_SPLIT_TILES, 1) > 0;
    if (!tiled || p.M < min_m || (ntiles < min_tiles && !split) || p.K % 128 ||
        (size_t)ntiles * kTileN * p.K / 2 >= (size_t(1) << 31) || (size_t)p.M * p.K * 4 >= (size_t(1) << 31))
        return -1;
    if (use_i4mm(ctx, p, ntiles, nsrc, xm))
        return st::int4_mm_f16(ctx, p.x, xm == XM_F32, p.perm, p.qw, p.sc, p.qz, p.zoff, p.y, p.M, p.K, p.N, p.gs, nsrc);
    const st::XsCall c{p.x, xm == XM_SILU ? p.xb : nullptr, xm == XM_F16, p.perm, {p.qw[0], p.qw[1]}, {p.sc[0], p.sc[1]},
                       {p.qz[0], p.qz[1]}, p.zoff, p.y, false, p.M, p.K, p.N, p.gs, nsrc, false, true};
    return st::int4_xs(ctx, c);
}

int launch_i4(st_context *ctx, QmvParams &p, bool tiled, int nsrc, int xm) {
    if (const int rc = launch_f16(ctx, p, tiled, nsrc, xm); rc != -1) return rc;
    p.units = p.K / p.gs;
    p.ntiles = (p.N + kTileN - 1) / kTileN;
    // the tiled kernels address the weights with 32-bit buffer offsets
    if (tiled && (size_t)p.ntiles * kTileN * p.K / 2 >= (size_t(1) << 31))
        return st::fail(ST_ERR_SHAPE, "qmv: tiled weight of %d x %d exceeds 2 GiB", p.K, p.N);
    if (tiled) return p.perm ? dispatch<FMT_I4T, true>(ctx, p, nsrc, xm) : dispatch<FMT_I4T, false>(ctx, p, nsrc, xm);
    return p.perm ? dispatch<FMT_I4, true>(ctx, p, nsrc, xm) : dispatch<FMT_I4, false>(ctx, p, nsrc, xm);
}

// Calls with more than kTokenBlock tokens that no f16-MFMA kernel takes run as
// blocks of kTokenBlock: the per-wave staging of the limb kernels grows with
// M * K per wave, and at 32 tokens two blocks of 16 (or eight of 4) measured
// several times faster than one launch, even though every block streams the
// weights again.
constexpr int kTokenBlock = 16;

// Fewest tokens for which st_int8_matvec takes the f16-MFMA kernel (f16 x, tiled weights).
constexpr int kI8mmMinM = 2;

template <typename F>
int by_token_blocks(const st_context *ctx, QmvParams &p, int xm, F &&launch) {
    const int blk = std::max(1, std::min(kTokenBlock, st::tune(ctx, ST_TUNE_TOKEN_BLOCK, kTokenBlock)));
    if (p.M <= blk) return launch(p);
    const size_t xe = xm == XM_F16 ? 2 : 4;
    for (int m0 = 0; m0 < p.M; m0 += blk) {
        QmvParams q = p;
        q.M = std::min(blk, p.M - m0);
        q.x = static_cast<const char *>(p.x) + (size_t)m0 * p.K * xe;
        if (p.xb) q.xb = p.xb + (size_t)m0 * p.K;
        q.y = p.y + (size_t)m0 * p.N;
        if (int rc = launch(q)) return rc;
    }
    return ST_OK;
}

// A GPTQ call of up to 32 tokens: one f16-MFMA launch when it is taken, else
// blocks of tokens (each of which may still be taken).
int launch_i4_blocks(st_context *ctx, QmvParams &p, bool tiled, int nsrc, int xm) {
    if (p.M > kTokenBlock && st::tune(ctx, ST_TUNE_TOKEN_BLOCK, 0) == 0)
        if (const int rc = launch_f16(ctx, p, tiled, nsrc, xm); rc != -1) return rc;
    return by_token_blocks(ctx, p, xm, [&](QmvParams &q) { return launch_i4(ctx, q, tiled, nsrc, xm); });
}

int check_i4(const char *fn, int M, int K, int N, int gs, int mmax) {
    if (gs != 64 && gs != 128 && gs != 256)
        return st::fail(ST_ERR_SHAPE, "%s: group_size %d not in {64,128,256}", fn, gs);
    if (M < 1 || M > mmax) return st::fail(ST_ERR_SHAPE, "%s: M=%d not in [1,%d]", fn, M, mmax);
    if (K <= 0 || K % gs) return st::fail(ST_ERR_SHAPE, "%s: K=%d not a positive multiple of group_size %d", fn, K, gs);
    if (N <= 0 || N % 8) return st::fail(ST_ERR_SHAPE, "%s: N=%d not a positive multiple of 8", fn, N);
    return ST_OK;
}

bool sc_ok(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 1) == 0; }

}  // namespace

extern "C" {

int st_gptq_i4_matvec(st_context *ctx, const void *x, int x_dtype, const uint32_t *qweight, const uint16_t *scales,
                      const uint32_t *qzeros, const int32_t *perm, float *y, int M, int K, int N, int group_size,
                      uint32_t flags) {
    if (!ctx || !x || !qweight || !scales || !y) return st::fail(ST_ERR_INVALID, "st_gptq_i4_matvec: NULL argument");
    if (int rc = check_i4("st_gptq_i4_matvec", M, K, N, group_size, 32)) return rc;
    if (!st::aligned16(qweight) || !st::aligned16(x) || !st::aligned16(perm) || !sc_ok(scales))
        return st::fail(ST_ERR_ALIGN, "st_gptq_i4_matvec: x/qweight/perm must be 16-byte aligned");
    if (x_dtype != ST_F32 && x_dtype != ST_F16) return st::fail(ST_ERR_INVALID, "st_gptq_i4_matvec: x_dtype %d", x_dtype);
    QmvParams p{};
    p.x = x;
    p.perm = perm;
    p.qw[0] = p.qw[1] = qweight;
    p.sc[0] = p.sc[1] = scales;
    p.qz[0] = p.qz[1] = qzeros;
    p.y = y;
    p.M = M;
    p.K = K;
    p.N = N;
    p.gs = group_size;
    p.zoff = (flags & ST_FLAG_ZEROS_PLUS_ONE) ? 1 : 0;
    const bool tiled = flags & ST_FLAG_TILED;
    const int xm = x_dtype == ST_F32 ? XM_F32 : XM_F16;
    return launch_i4_blocks(ctx, p, tiled, 1, xm);
}

int st_gptq_i4_matvec_noalloc(st_context *ctx, const void *x, int x_dtype, const uint32_t *qweight,
                              const uint16_t *scales, const uint32_t *qzeros, const int32_t *perm, float *y, int M,
                              int K, int N, int group_size, uint32_t flags) {
    if (!ctx) return st::fail(ST_ERR_INVALID, "st_gptq_i4_matvec_noalloc: ctx is NULL");
    if (!ctx->scratch) return st::fail(ST_ERR_WORKSPACE, "st_gptq_i4_matvec_noalloc: no scratch on this device");
    // The most any path of the call keeps: i4mm's pre-pass rows of f32 x (2 f16
    // rows per token and a factor per 128 k; the skinny kernel's gathered f32 x
    // is smaller) or, for f16 x under act-order, the gathered rows. f32 x without
    // act-order keeps none of it unless I4MM_PREPASS is set, but is held to the
    // same limit. Split-K partials shrink (or go unsplit) to fit what is there.
    if (M > 0 && K > 0 && (x_dtype == ST_F32 || perm)) {
        // (f16 x under act-order: the gathered rows, mb K halves)
        const size_t mb = (size_t)std::min(M, 2 * kTokenBlock);
        const size_t need = x_dtype == ST_F32 ? 2 * mb * K * 2 + mb * (size_t)(K / 128) * 4 : mb * K * 2;
        if (need > ST_NOALLOC_SCRATCH_BYTES)
            return st::fail(ST_ERR_WORKSPACE, "st_gptq_i4_matvec_noalloc: %zu bytes of scratch needed, %u held", need,
                            (unsigned)ST_NOALLOC_SCRATCH_BYTES);
    }
    st_context view = *ctx;  // the same stream and settings, the scratch as workspace
    view.ws = static_cast<float *>(ctx->scratch);
    view.ws_bytes = ST_NOALLOC_SCRATCH_BYTES;
    view.own_stream = false;
    return st_gptq_i4_matvec(&view, x, x_dtype, qweight, scales, qzeros, perm, y, M, K, N, group_size, flags);
}

int st_gptq_i4_silu_matvec(st_context *ctx, const float *a, const float *b, const uint32_t *qweight,
                           const uint16_t *scales, const uint32_t *qzeros, const int32_t *perm, float *y, int M, int K,
                           int N, int group_size, uint32_t flags) {
    if (!ctx || !a || !b || !qweight || !scales || !y)
        return st::fail(ST_ERR_INVALID, "st_gptq_i4_silu_matvec: NULL argument");
    if (int rc = check_i4("st_gptq_i4_silu_matvec", M, K, N, group_size, 32)) return rc;
    if (!st::aligned16(qweight) || !st::aligned16(a) || !st::aligned16(b) || !st::aligned16(perm) || !sc_ok(scales))
        return st::fail(ST_ERR_ALIGN, "st_gptq_i4_silu_matvec: a/b/qweight/perm must be 16-byte aligned");
    QmvParams p{};
    p.x = a;
    p.xb = b;
    p.perm = perm;
    p.qw[0] = p.qw[1] = qweight;
    p.sc[0] = p.sc[1] = scales;
    p.qz[0] = p.qz[1] = qzeros;
    p.y = y;
    p.M = M;
    p.K = K;
    p.N = N;
    p.gs = group_size;
    p.zoff = (flags & ST_FLAG_ZEROS_PLUS_ONE) ? 1 : 0;
    const bool tiled = flags & ST_FLAG_TILED;
    return launch_i4_blocks(ctx, p, tiled, 1, XM_SILU);
}

int st_gptq_i4_gate_up_silu(st_context *ctx, const void *x, int x_dtype, const uint32_t *qweight_gate,
                            const uint16_t *scales_gate, const uint32_t *qzeros_gate, const uint32_t *qweight_up,
                            const uint16_t *scales_up, const uint32_t *qzeros_up, const int32_t *perm, float *y, int M,
                            int K, int N, int group_size, uint32_t flags) {
    if (!ctx || !x || !qweight_gate || !scales_gate || !qweight_up || !scales_up || !y)
        return st::fail(ST_ERR_INVALID, "st_gptq_i4_gate_up_silu: NULL argument");
    if (int rc = check_i4("st_gptq_i4_gate_up_silu", M, K, N, group_size, 32)) return rc;
    if ((qzeros_gate == nullptr) != (qzeros_up == nullptr))
        return st::fail(ST_ERR_INVALID, "st_gptq_i4_gate_up_silu: give qzeros for both or neither");
    if (!st::aligned16(qweight_gate) || !st::aligned16(qweight_up) || !st::aligned16(x) || !st::aligned16(perm) ||
        !sc_ok(scales_gate) || !sc_ok(scales_up))
        return st::fail(ST_ERR_ALIGN, "st_gptq_i4_gate_up_silu: x/qweight/perm must be 16-byte aligned");
    if (x_dtype != ST_F32 && x_dtype != ST_F16)
        return st::fail(ST_ERR_INVALID, "st_gptq_i4_gate_up_silu: x_dtype %d", x_dtype);
    QmvParams p{};
    p.x = x;
    p.perm = perm;
    p.qw[0] = qweight_gate;
    p.qw[1] = qweight_up;
    p.sc[0] = scales_gate;
    p.sc[1] = scales_up;
    p.qz[0] = qzeros_gate;
    p.qz[1] = qzeros_up;
    p.y = y;
    p.M = M;
    p.K = K;
    p.N = N;
    p.gs = group_size;
    p.zoff = (flags & ST_FLAG_ZEROS_PLUS_ONE) ? 1 : 0;
    const bool tiled = flags & ST_FLAG_TILED;
    const int xm = x_dtype == ST_F32 ? XM_F32 : XM_F16;
    return launch_i4_blocks(ctx, p, tiled, 2, xm);
}

size_t st_gptq_i4_tiled_words(int K, int N, int group_size) {
    if (K <= 0 || N <= 0 || group_size <= 0 || K % group_size) return 0;
    return (size_t)((N + kTileN - 1) / kTileN) * kTileN * (size_t)(K / 8);
}

int st_gptq_i4_repack(st_context *ctx, const uint32_t *qweight, uint32_t *qweight_tiled, int K, int N,
                      int group_size) {
    if (!ctx || !qweight || !qweight_tiled) return st::fail(ST_ERR_INVALID, "st_gptq_i4_repack: NULL argument");
    if (int rc = check_i4("st_gptq_i4_repack", 1, K, N, group_size, 1)) return rc;
    if (!st::aligned16(qweight_tiled))
        return st::fail(ST_ERR_ALIGN, "st_gptq_i4_repack: output must be 16-byte aligned");
    const int ntiles = (N + kTileN - 1) / kTileN;
    const long long total = (long long)ntiles * (K / group_size) * 64 * (group_size / 32);
    st::launch(ctx, repack_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, qweight,
                       qweight_tiled, K, N, group_size, ntiles);
    return st::launch_check("repack_kernel");
}

size_t st_int8_tiled_bytes(int K, int N) {
    if (K <= 0 || N <= 0) return 0;
    return (size_t)((N + kTileN - 1) / kTileN) * kTileN * (size_t)K;
}

int st_int8_repack(st_context *ctx, const int8_t *w, int8_t *w_tiled, int K, int N) {
    if (!ctx || !w || !w_tiled) return st::fail(ST_ERR_INVALID, "st_int8_repack: NULL argument");
    if (K <= 0 || K % 128 || N <= 0) return st::fail(ST_ERR_SHAPE, "st_int8_repack: K=%d (multiple of 128), N=%d", K, N);
    if (!st::aligned16(w) || !st::aligned16(w_tiled))
        return st::fail(ST_ERR_ALIGN, "st_int8_repack: w and w_tiled must be 16-byte aligned");
    const int ntiles = (N + kTileN - 1) / kTileN;
    const long long total = (long long)ntiles * (K / 128) * 128;
    st::launch(ctx, repack8_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, w, w_tiled, K,
                       N, ntiles);
    return st::launch_check("repack8_kernel");
}

int st_int8_matvec(st_context *ctx, const void *x, int x_dtype, const int8_t *w, const float *scale, float *y, int M,
                   int K, int N, uint32_t flags) {
    if (!ctx || !x || !w || !scale || !y) return st::fail(ST_ERR_INVALID, "st_int8_matvec: NULL argument");
    if (M < 1 || M > 32) return st::fail(ST_ERR_SHAPE, "st_int8_matvec: M=%d not in [1,32]", M);
    if (K <= 0 || K % 128) return st::fail(ST_ERR_SHAPE, "st_int8_matvec: K=%d not a positive multiple of 128", K);
    if (N <= 0 || N % 4) return st::fail(ST_ERR_SHAPE, "st_int8_matvec: N=%d not a positive multiple of 4", N);
    const bool tiled = (flags & ST_FLAG_TILED) != 0;
    if ((long long)((N + kTileN - 1) / kTileN) * kTileN * K >= (1ll << 31))  // 32-bit buffer offsets
        return st::fail(ST_ERR_SHAPE, "st_int8_matvec: weight of %d x %d exceeds 2 GiB", N, K);
    if (!st::aligned16(w) || !st::aligned16(x))
        return st::fail(ST_ERR_ALIGN, "st_int8_matvec: w and x must be 16-byte aligned");
    if (x_dtype != ST_F32 && x_dtype != ST_F16) return st::fail(ST_ERR_INVALID, "st_int8_matvec: x_dtype %d", x_dtype);
    // Several tokens with f16 x on tiled weights: the f16-MFMA skinny GEMM,
    // which reads the weights once for all tokens.
    if (tiled && x_dtype == ST_F16 && M >= st::tune(ctx, ST_TUNE_I8MM_MIN_M, kI8mmMinM))
        return st::int8_mm_f16(ctx, x, w, scale, y, M, K, N);
    QmvParams p{};
    p.x = x;
    p.w8 = w;
    p.scale8 = scale;
    p.y = y;
    p.M = M;
    p.K = K;
    p.N = N;
    p.gs = 128;
    p.units = K / 128;
    p.ntiles = (N + kTileN - 1) / kTileN;
    const int xm = x_dtype == ST_F32 ? XM_F32 : XM_F16;
    return by_token_blocks(ctx, p, xm, [&](QmvParams &q) {
        return tiled ? dispatch<FMT_I8T, false>(ctx, q, 1, xm) : dispatch<FMT_I8, false>(ctx, q, 1, xm);
    });
}

}  // extern "C"
