"""The skinny GPTQ kernel (csrc/i4xs.hpp: x in registers, several tokens)
through the entry points that take it, against the f64 oracle, at the edges
of its tiles and splits: 16 / 32-token blocks, waves with no unit or one unit
less (K of one unit up to 32 per workgroup), K slices across workgroups,
ragged last tiles, every group size, zero points, act-order, silu(a) * b."""
import numpy as np
import pytest
import torch

import shady_thinker_amd as sta
from shady_thinker_amd import model as M
from shady_thinker_amd._lib import launches

pytestmark = pytest.mark.gpu

# Bounds. x is held to 2^-22 of itself or better and every product is exact,
# so what is left are f32 sums: of 128 products inside the MFMA and of at most
# a few hundred groups after it, errors of both signs: below 2^-20.
TOL = 1e-6
# One rounding to f16 of every weight or product: at most 2^-11 each, of both
# signs, 2^-11 / sqrt(3) rms at worst.
TOL_F16 = 3e-4


def _case(orc, seed, K, N, gs, zeros, act, Mr, f16):
    return orc.gptq_case(seed, K, N, gs, zeros=zeros, act_order=act, M=Mr, x_dtype=np.float16 if f16 else np.float32)


def _up(gpu, c, gs):
    return sta.GptqWeight.upload(gpu, c["qweight"], c["scales"], gs, qzeros=c["qzeros"], g_idx=c["g_idx"])


def _ref(orc, c, x, K, N, gs, act):
    return orc.gptq_matvec_f64(x, c["qweight"], c["scales"], K, N, gs, qzeros=c["qzeros"],
                               g_idx=c["g_idx"] if act else None)


@pytest.mark.parametrize("Mr,K,N,gs,zeros,act,f16", [
    (9, 128, 24, 128, False, False, False),      # one unit: seven waves without one; a ragged tile
    (16, 1152, 4120, 128, True, False, False),   # nine units: one wave with two
    (17, 2560, 8208, 128, False, False, False),  # two token blocks, units 3 and 2, 513 tiles
    (31, 4096, 264, 64, True, False, False),     # four units a wave, group 64
    (32, 4352, 1032, 256, False, False, False),  # more than 32 units: K slices, group 256 split inside a group
    (11, 11008, 520, 128, True, False, False),   # 86 units
    (5, 2048, 2056, 128, False, False, False),   # fewest tokens on narrow linears
    (3, 3072, 1032, 128, True, True, False),     # act-order: fewest tokens
    (24, 4096, 4104, 64, True, True, False),     # act-order, group 64, 257 tiles
    (7, 2560, 13000, 128, False, False, False),  # one source of more than 3 tiles per CU
    (8, 1024, 8192, 64, True, True, False),      # group 64, two tiles per CU: the last of its rule
    (5, 3072, 8200, 64, False, False, False),    # one tile more
    (20, 1024, 4112, 128, True, False, True),    # f16 x, one token block
    (32, 6144, 776, 64, True, True, True),       # f16 x gathered
])
def test_skinny_matvec(gpu, orc, Mr, K, N, gs, zeros, act, f16):
    c = _case(orc, 700 + Mr + K, K, N, gs, zeros, act, Mr, f16)
    w = _up(gpu, c, gs)
    x = torch.from_numpy(c["x"]).cuda()
    y = torch.full((Mr, N), float("nan"), device="cuda")
    M.gptq_matvec(gpu, "t", x, w.qweight, w.scales, y, K, N, gs, w.qzeros, w.perm, w.flags)
    torch.cuda.synchronize()
    assert orc.rel_l2(y.cpu().numpy(), _ref(orc, c, c["x"], K, N, gs, act)) < TOL


@pytest.mark.parametrize("Mr,K,N,gs,zeros,act", [
    (22, 11008, 1416, 128, False, True),
    (10, 10240, 2488, 128, True, False),
    (26, 9472, 624, 256, False, False),
])
def test_skinny_f32_sums(gpu, orc, Mr, K, N, gs, zeros, act):
    """f32 x keeps f32 sums: the hi parts' products (nearly exact in f32) and the
    lo parts' are summed apart within a group, and the groups in few roundings.

    Bound: x is held to half a unit of its 22nd bit or better, 2^-23 / sqrt(3)
    = 6.9e-8 rms at the worst mantissa and 4.6e-8 over a binade. After it a sum
    is rounded at most 4 times within a wave, 3 over the waves and 4 over the
    slices, each 2^-24 / sqrt(3) = 3.4e-8 of the sum so far (sqrt(j / n) of the
    whole one after j of n equal parts): sqrt(2.5 + 1.75 + 1.9) 3.4e-8 = 8.5e-8
    in all, 9.7e-8 with x's part. (In one chain of hi and lo: 1.34e-7.)"""
    c = _case(orc, 1100 + Mr, K, N, gs, zeros, act, Mr, False)
    w = _up(gpu, c, gs)
    y = torch.full((Mr, N), float("nan"), device="cuda")
    launches()
    M.gptq_matvec(gpu, "t", torch.from_numpy(c["x"]).cuda(), w.qweight, w.scales, y, K, N, gs, w.qzeros, w.perm, w.flags)
    assert "i4xs_kernel" in launches()
    torch.cuda.synchronize()
    assert orc.rel_l2(y.cpu().numpy(), _ref(orc, c, c["x"], K, N, gs, act)) < 1.1e-7


@pytest.mark.parametrize("Mr,K,N,gs,zeros,act", [
    (5, 1024, 264, 128, False, False),
    (16, 2048, 2568, 128, True, False),
    (31, 4096, 1032, 64, False, False),   # K slices (two units a wave at most)
    (9, 3072, 520, 256, True, True),      # act-order: the product is gathered
])
def test_skinny_silu_matvec(gpu, orc, Mr, K, N, gs, zeros, act):
    c = _case(orc, 800 + Mr, K, N, gs, zeros, act, Mr, False)
    w = _up(gpu, c, gs)
    rng = np.random.default_rng(Mr)
    a, b = (rng.standard_normal((Mr, K)).astype(np.float32) for _ in range(2))
    y = torch.full((Mr, N), float("nan"), device="cuda")
    M.fused_silu_gptq_down(gpu, torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda(), w.qweight, w.scales, y, K, N, gs,
                           w.qzeros, w.perm, w.flags)
    torch.cuda.synchronize()
    # (the hardware exp and division of silu: a few ulp of f32)
    assert orc.rel_l2(y.cpu().numpy(), _ref(orc, c, orc.silu_gate_f64(a, b), K, N, gs, act)) < 2e-6


@pytest.mark.parametrize("Mr,K,N,gs,zeros,act,f16", [
    (9, 1536, 4120, 128, True, False, False),
    (32, 4096, 1032, 64, False, False, False),
    (17, 5120, 776, 256, True, True, True),
    (12, 3328, 1032, 64, True, False, False),  # group 64 with zero points: two units a wave, K slices
    (32, 2304, 14336, 64, True, False, False),  # three (many columns of two token blocks): K in one piece
    (27, 2560, 13064, 64, True, True, True),
])
def test_skinny_gate_up(gpu, orc, Mr, K, N, gs, zeros, act, f16):
    c = _case(orc, 900 + Mr, K, N, gs, zeros, act, Mr, f16)
    c2 = _case(orc, 950 + Mr, K, N, gs, zeros, act, Mr, f16)
    c2["g_idx"] = c["g_idx"]
    g, u = _up(gpu, c, gs), _up(gpu, c2, gs)
    x = torch.from_numpy(c["x"]).cuda()
    y = torch.full((Mr, N), float("nan"), device="cuda")
    launches()
    M.fused_gate_up_silu(gpu, x, g.qweight, g.scales, u.qweight, u.scales, y, K, N, gs, gate_qz=g.qzeros, up_qz=u.qzeros,
                         perm=g.perm, flags=g.flags)
    ran = launches()
    assert "i4xs_kernel" in ran and (N < 13064 or "i4xs_reduce_kernel" not in ran)
    torch.cuda.synchronize()
    ref = orc.silu_gate_f64(_ref(orc, c, c["x"], K, N, gs, act), _ref(orc, c2, c["x"], K, N, gs, act))
    assert orc.rel_l2(y.cpu().numpy(), ref) < 3e-6  # silu and the product add their own f32 steps


@pytest.mark.parametrize("Mr,K,N,gs,zeros,act,silu,out", [
    (33, 1024, 264, 128, False, False, False, torch.float32),
    (64, 2560, 4104, 128, True, False, False, torch.float32),
    (97, 4096, 1032, 64, True, True, False, torch.float16),
    (160, 11008, 520, 128, False, False, False, torch.float16),
    (256, 1280, 2056, 256, True, False, False, torch.float32),
    (161, 1024, 16392, 128, False, False, False, torch.float32),  # past the rule: the GEMM
    (1, 2048, 136, 128, True, False, False, torch.float32),
    (77, 4096, 520, 128, True, False, True, torch.float32),
    (40, 1152, 1032, 64, False, False, True, torch.float16),
    (100, 9728, 520, 64, True, True, True, torch.float16),  # act-order: the product is gathered
    (33, 32768, 24, 256, False, False, True, torch.float32),  # the longest row of the product's pre-pass
    (35, 8320, 264, 128, True, True, True, torch.float32),  # 8 k past a pass of its threads
])
def test_skinny_gemm(gpu, orc, Mr, K, N, gs, zeros, act, silu, out):
    c = _case(orc, 1000 + Mr, K, N, gs, zeros, act, Mr, True)
    w = _up(gpu, c, gs)
    x = torch.from_numpy(c["x"]).cuda()
    y = torch.full((Mr, N), float("nan"), device="cuda", dtype=out)
    if silu:
        b = np.random.default_rng(Mr).standard_normal((Mr, K)).astype(np.float16)
        M.fused_silu_gptq_gemm(gpu, x, torch.from_numpy(b).cuda(), w.qweight, w.scales, y, K, N, gs, w.qzeros, w.perm,
                               w.flags)
        xin = orc.silu_gate_f64(c["x"], b)
    else:
        M.gptq_gemm(gpu, x, w.qweight, w.scales, y, K, N, gs, w.qzeros, w.perm, w.flags)
        xin = c["x"]
    torch.cuda.synchronize()
    # weights (silu: the product) rounded once to f16, then C
    tol = TOL_F16 * (2**0.5 if out == torch.float16 else 1)
    assert orc.rel_l2(y.float().cpu().numpy(), _ref(orc, c, xin, K, N, gs, act)) < tol


@pytest.mark.parametrize("Mr,K,N,gs,act", [(77, 4096, 520, 128, True), (40, 9728, 264, 64, True), (64, 2048, 264, 128, False)])
def test_skinny_gate_up_gemm(gpu, orc, Mr, K, N, gs, act):
    """Gate and up of a short prompt: x gathered once for both weights, results
    those of two single calls."""
    c = _case(orc, 1150, K, N, gs, False, act, Mr, True)
    c2 = _case(orc, 1151, K, N, gs, False, act, Mr, True)
    c2["g_idx"] = c["g_idx"]
    ws = [_up(gpu, v, gs) for v in (c, c2)]
    x = torch.from_numpy(c["x"]).cuda()
    y = [torch.full((Mr, N), float("nan"), device="cuda") for _ in range(4)]
    launches()
    M.gate_up_gemm(gpu, x, ws[0].qweight, ws[0].scales, ws[1].qweight, ws[1].scales, y[0], y[1], K, N, gs, perm=ws[0].perm,
                   flags=ws[0].flags)
    ran = launches()
    assert ran.count("i4xs_kernel") == 2 and ran.count("i4xs_gather_kernel") == int(act)
    for w, o in zip(ws, y[2:]):
        M.gptq_gemm(gpu, x, w.qweight, w.scales, o, K, N, gs, None, w.perm, w.flags)
    torch.cuda.synchronize()
    assert torch.equal(y[0], y[2]) and torch.equal(y[1], y[3])
    assert orc.rel_l2(y[1].cpu().numpy(), _ref(orc, c2, c["x"], K, N, gs, act)) < TOL_F16


def test_skinny_gemm_silu_scales(gpu, orc):
    """f16 silu(a) * b of very different size by token: past f16's range, below
    its normals, zero, and one that is not finite, each row by itself."""
    Mr, K, N = 36, 2176, 264
    c = _case(orc, 81, K, N, 128, False, False, Mr, True)
    w = _up(gpu, c, 128)
    rng = np.random.default_rng(81)
    a, b = (rng.standard_normal((Mr, K)) for _ in range(2))
    size = 2.0 ** np.linspace(-12, 11, Mr)
    a, b = (a * size[:, None]).astype(np.float16), (b * size[:, None]).astype(np.float16)
    a[5], b[7, 3] = 0, np.inf
    y = torch.full((Mr, N), float("nan"), device="cuda")
    M.fused_silu_gptq_gemm(gpu, torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda(), w.qweight, w.scales, y, K, N, 128,
                           w.qzeros, w.perm, w.flags)
    torch.cuda.synchronize()
    y = y.cpu().numpy().astype(np.float64)
    assert not y[5].any() and not np.isfinite(y[7]).any()
    keep = [i for i in range(Mr) if i not in (5, 7)]
    ref = _ref(orc, c, orc.silu_gate_f64(a[keep], b[keep]), K, N, 128, False)
    for i, r in zip(keep, ref):
        assert orc.rel_l2(y[i] / np.abs(r).max(), r / np.abs(r).max()) < TOL_F16, i


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_skinny_nonfinite_row(gpu, orc, bad):
    """A NaN or infinity in one token poisons that token's row only."""
    Mr, K, N = 18, 2560, 264
    c = _case(orc, 77, K, N, 128, False, False, Mr, False)
    w = _up(gpu, c, 128)
    x = c["x"].copy()
    x[3, 1000] = bad
    y = torch.zeros(Mr, N, device="cuda")
    M.gptq_matvec(gpu, "t", torch.from_numpy(x).cuda(), w.qweight, w.scales, y, K, N, 128, flags=w.flags)
    torch.cuda.synchronize()
    y = y.cpu().numpy()
    assert not np.isfinite(y[3]).any()
    keep = [i for i in range(Mr) if i != 3]
    ref = _ref(orc, c, c["x"], K, N, 128, False)
    assert orc.rel_l2(y[keep], ref[keep]) < TOL


def test_skinny_scales_of_x(gpu, orc):
    """Rows of very different size, zero rows, values down to f32's smallest
    normals beside large ones: each row within the bound by itself."""
    Mr, K, N = 16, 2560, 264
    c = _case(orc, 78, K, N, 128, True, False, Mr, False)
    w = _up(gpu, c, 128)
    x = c["x"] * (np.float32(10.0) ** np.linspace(-34, 30, Mr).astype(np.float32))[:, None]
    x[5] = 0.0
    x[7, :1280] *= np.float32(1e-7)
    x = x.astype(np.float32)
    y = torch.full((Mr, N), float("nan"), device="cuda")
    M.gptq_matvec(gpu, "t", torch.from_numpy(x).cuda(), w.qweight, w.scales, y, K, N, 128, w.qzeros, None, w.flags)
    torch.cuda.synchronize()
    y = y.cpu().numpy()
    ref = _ref(orc, c, x, K, N, 128, False)
    assert not y[5].any()
    for r in range(Mr):
        if r != 5:
            assert orc.rel_l2(y[r].astype(np.float64) / np.abs(ref[r]).max(), ref[r] / np.abs(ref[r]).max()) < TOL, r


def test_skinny_graph_replay(gpu, orc):
    """Two calls with K slices in the workspace, captured: every replay equals eager."""
    Mr, K, N = 20, 9728, 520
    c = _case(orc, 79, K, N, 128, False, False, Mr, False)
    w = _up(gpu, c, 128)
    x = torch.from_numpy(c["x"]).cuda()
    y, z = torch.empty(Mr, N, device="cuda"), torch.empty(Mr, N, device="cuda")

    def calls():
        for o in (y, z):
            M.gptq_matvec(gpu, "t", x, w.qweight, w.scales, o, K, N, 128, flags=w.flags)

    calls()
    torch.cuda.synchronize()
    eager = y.clone()
    s, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(s), torch.cuda.graph(g, stream=s):
        calls()
    for _ in range(3):
        y.zero_(), z.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, eager) and torch.equal(z, eager)
        M.gptq_matvec(gpu, "t", x, w.qweight, w.scales, y, K, N, 128, flags=w.flags)  # eager work between
        torch.cuda.synchronize()
