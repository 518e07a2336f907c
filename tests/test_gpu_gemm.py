"""GPU parity of the prefill GEMM st_gptq_i4_gemm against the CPU oracle and
a torch fp32 reference, through the C ABI.

Bar: GEMM outputs within rel-L2 2e-3. The kernel
forms (q - z) exactly and rounds (q - z) * s once to f16 per weight, then
accumulates in f32 on MFMA; so it is checked three ways: against the f64
oracle (bar 2e-3; typically ~2e-4), bit for bit on one-hot rows and integer
cases (where it must equal the f16-rounded dequant), and against a torch fp32
matmul over those f16-rounded weights (accumulation order only, ~1e-6).
"""
import numpy as np
import pytest
import torch

import shady_thinker_amd as sta
from shady_thinker_amd import model as M
from shady_thinker_amd._lib import launches

pytestmark = pytest.mark.gpu

TOL = 2e-3  # rel-L2, prefill GEMM (north_star)


def up(gpu, case, zeros_plus_one=False, tiled=True):
    return sta.GptqWeight.upload(gpu, case["qweight"], case["scales"], case["gs"], qzeros=case["qzeros"],
                                 g_idx=case["g_idx"], zeros_plus_one=zeros_plus_one, tiled=tiled)


def run_gemm(gpu, w, a_np, out_dtype=torch.float32):
    a = torch.from_numpy(np.ascontiguousarray(a_np, dtype=np.float16)).to(gpu.device)
    c = torch.empty(a.shape[0], w.N, dtype=out_dtype, device=gpu.device)
    M.gptq_gemm(gpu, a, w.qweight, w.scales, c, w.K, w.N, w.group_size, w.qzeros, w.perm, w.flags)
    torch.cuda.synchronize()
    return c.float().cpu().numpy()


# Short prompts on tiled weights go to the skinny kernel (i4xs.hpp). Tests of
# the GEMM at such sizes run twice: as dispatched, and with GEMM_CB set, which
# keeps the skinny kernel out (0: the GEMM's tile stays its own choice).
@pytest.fixture(params=["skinny", "gemm"])
def route(request, tune):
    if request.param == "gemm":
        tune(GEMM_CB=0)
    launches()
    yield request.param
    ran = set(launches())
    assert ("gemm_kernel" in ran, "i4xs_kernel" in ran) == (request.param == "gemm", request.param == "skinny")


@pytest.mark.parametrize("tiled", [True, False])
@pytest.mark.parametrize("Mr,K,N,gs,zeros,act", [
    (1, 256, 64, 128, False, False),
    (33, 512, 200, 128, False, False),
    (130, 1024, 264, 64, True, False),
    (257, 2048, 520, 256, False, True),
    (96, 1024, 136, 128, True, True),
    (129, 768, 384, 64, False, True),
])
def test_gemm_matches_oracle(gpu, orc, tiled, Mr, K, N, gs, zeros, act):
    c = orc.gptq_case(10 + Mr, K, N, gs, zeros=zeros, act_order=act, M=Mr, x_dtype=np.float16)
    w = up(gpu, c, tiled=tiled)
    y = run_gemm(gpu, w, c["x"])
    ref = orc.gptq_matvec_f64(c["x"], c["qweight"], c["scales"], K, N, gs, qzeros=c["qzeros"], g_idx=c["g_idx"])
    e = orc.rel_l2(y, ref)
    print(f"gemm M={Mr} K={K} N={N} gs={gs} zeros={zeros} act={act} tiled={tiled}: rel-L2 {e:.3e}")
    assert e < TOL
    assert e < 5e-4  # one f16 rounding per weight: ~2e-4


@pytest.mark.parametrize("tiled", [True, False])
def test_gemm_f16_output_and_zeros_plus_one(gpu, orc, tiled):
    Mr, K, N, gs = 200, 1024, 328, 128
    c = orc.gptq_case(5, K, N, gs, zeros=True, M=Mr, x_dtype=np.float16)
    w = up(gpu, c, zeros_plus_one=True, tiled=tiled)
    y = run_gemm(gpu, w, c["x"], torch.float16)
    ref = orc.gptq_matvec_f64(c["x"], c["qweight"], c["scales"], K, N, gs, qzeros=c["qzeros"], zero_offset=1)
    e = orc.rel_l2(y, ref)
    print(f"gemm f16 out, zeros+1: rel-L2 {e:.3e}")
    assert e < TOL


@pytest.mark.parametrize("tiled", [True, False])
def test_gemm_one_hot_rows_are_dequant_rows(gpu, orc, tiled):
    K, N, gs = 1024, 264, 128
    c = orc.gptq_case(1, K, N, gs, zeros=True)
    w = up(gpu, c, tiled=tiled)
    W = orc.gptq_dequant_f32(c["qweight"], c["scales"], K, N, gs, qzeros=c["qzeros"])
    ks = [0, 1, 7, 8, 63, 64, 127, 128, 500, 1023] * 4  # 40 rows: more than one MFMA block
    a = np.zeros((len(ks), K), np.float16)
    for i, k in enumerate(ks):
        a[i, k] = 1.0
    y = run_gemm(gpu, w, a)
    W16 = W.astype(np.float16).astype(np.float32)  # (q - z) * s rounded once to f16
    assert np.array_equal(y, W16[ks]), "one-hot rows must be the f16-rounded dequant, bit for bit"


def test_gemm_integer_case_bit_equal(gpu, orc):
    Mr, K, N, gs = 64, 2048, 256, 128
    c = orc.gptq_case(2, K, N, gs, zeros=True, act_order=True)
    c["scales"] = np.ones_like(c["scales"])
    rng = np.random.default_rng(3)
    a = rng.integers(-3, 4, size=(Mr, K)).astype(np.float16)
    w = up(gpu, c)
    y = run_gemm(gpu, w, a)
    ref = orc.gptq_matvec_f64(a, c["qweight"], c["scales"], K, N, gs, qzeros=c["qzeros"], g_idx=c["g_idx"])
    assert np.array_equal(y.astype(np.float64), ref)


def test_gemm_agrees_with_decode_on_shared_rows(gpu, orc):
    """linear() sends M <= 32 to the matvec and M > 32 to the GEMM; the two
    must agree on the same weights (both are exact-dequant, f32-accumulate)."""
    K, N, gs = 2048, 512, 128
    c = orc.gptq_case(4, K, N, gs, act_order=True, M=48, x_dtype=np.float16)
    w = up(gpu, c)
    x = torch.from_numpy(c["x"]).to(gpu.device)
    y_g = torch.empty(48, N, device=gpu.device)
    sta.linear(gpu, x, w, y_g)
    y_m = torch.empty(16, N, device=gpu.device)
    sta.linear(gpu, x[:16].contiguous(), w, y_m)
    torch.cuda.synchronize()
    e = orc.rel_l2(y_g[:16].cpu().numpy(), y_m.cpu().numpy())
    assert e < 1e-3  # matvec: exact dequant; GEMM: one f16 rounding per weight


@pytest.mark.parametrize("Mr", [512, 2048])
def test_gemm_full_config_vs_oracle(gpu, orc, Mr):
    """configs[3] at full size (M in {512, 2048}, K=4096, N=14336, g128,
    act-order, tiled weights uploaded as a checkpoint would be), with
    references that do not go through the HIP path:
    * the f64 oracle on three 256-column slices (columns are independent:
      the slice's qweight and scales give exactly those outputs), bar 2e-3;
    * torch fp32 over the oracle's exact f32 dequant of the whole matrix
      (rows in checkpoint order, groups through g_idx): rel-L2 below 5e-4;
    * the same over that dequant rounded to f16, which is what the kernel
      multiplies: rel-L2 below 1e-5 (accumulation order only)."""
    K, N, gs = 4096, 14336, 128
    c = orc.gptq_case(700 + Mr // 512, K, N, gs, act_order=True, M=Mr, x_dtype=np.float16)
    w = up(gpu, c)
    y = run_gemm(gpu, w, c["x"])
    for n0 in (0, 7040, N - 256):
        qw = np.ascontiguousarray(c["qweight"][:, n0:n0 + 256])
        sc = np.ascontiguousarray(c["scales"][:, n0:n0 + 256])
        ref = orc.gptq_matvec_f64(c["x"], qw, sc, K, 256, gs, g_idx=c["g_idx"])
        e = orc.rel_l2(y[:, n0:n0 + 256], ref)
        print(f"configs[3] M={Mr} columns {n0}..{n0 + 255}: rel-L2 {e:.3e} vs f64")
        assert e < TOL
    W = torch.from_numpy(orc.gptq_dequant_f32(c["qweight"], c["scales"], K, N, gs, g_idx=c["g_idx"])).to(gpu.device)
    A = torch.from_numpy(c["x"]).to(gpu.device).float()
    C = torch.from_numpy(y).to(gpu.device)
    rel = lambda ref: (torch.linalg.vector_norm((C - ref).double()) / torch.linalg.vector_norm(ref.double())).item()
    e = rel(A @ W)
    e16 = rel(A @ W.half().float())
    print(f"configs[3] M={Mr} vs torch fp32: rel-L2 {e:.3e} (exact dequant), {e16:.3e} (f16-rounded dequant)")
    assert e < 5e-4
    assert e16 < 1e-5


def test_gemm_graph_replay_matches_eager(gpu, orc, route):
    Mr, K, N, gs = 160, 1024, 392, 128
    c = orc.gptq_case(8, K, N, gs, act_order=True, M=Mr, x_dtype=np.float16)
    w = up(gpu, c)
    a = torch.from_numpy(c["x"]).to(gpu.device)
    eager = torch.empty(Mr, N, device=gpu.device)
    M.gptq_gemm(gpu, a, w.qweight, w.scales, eager, K, N, gs, w.qzeros, w.perm, w.flags)
    torch.cuda.synchronize()
    out = torch.empty_like(eager)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        M.gptq_gemm(gpu, a, w.qweight, w.scales, out, K, N, gs, w.qzeros, w.perm, w.flags)  # warm on s
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            M.gptq_gemm(gpu, a, w.qweight, w.scales, out, K, N, gs, w.qzeros, w.perm, w.flags)
    for i in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), f"replay {i}"
        M.gptq_gemm(gpu, a, w.qweight, w.scales, eager, K, N, gs, w.qzeros, w.perm, w.flags)  # eager work between
        torch.cuda.synchronize()


@pytest.mark.parametrize("gs", [64, 128, 256])
def test_gemm_split_k_matches_unsplit(gpu, orc, gs, tune):
    """Small grids split K across workgroups (f32 partials in the context
    workspace, reduced in a fixed order): same result as one workgroup per
    tile up to summation order, and the oracle's."""
    Mr, K, N = 64, 4096, 264
    c = orc.gptq_case(60 + gs, K, N, gs, zeros=True, act_order=True, M=Mr, x_dtype=np.float16)
    w = up(gpu, c)
    tune(GEMM_CB=0)  # (else the skinny kernel takes so few rows)
    launches()
    y_split = run_gemm(gpu, w, c["x"])
    assert "splitk_reduce_kernel" in launches()
    tune(GEMM_NO_SPLIT=1)
    y_one = run_gemm(gpu, w, c["x"])
    assert launches()[-1] == "gemm_kernel"
    ref = orc.gptq_matvec_f64(c["x"], c["qweight"], c["scales"], K, N, gs, qzeros=c["qzeros"], g_idx=c["g_idx"])
    e_s, e_o, e_so = orc.rel_l2(y_split, ref), orc.rel_l2(y_one, ref), orc.rel_l2(y_split, y_one)
    print(f"split-K gs={gs}: split {e_s:.3e}, one {e_o:.3e}, split vs one {e_so:.3e}")
    assert e_s < 5e-4 and e_o < 5e-4 and e_so < 1e-5


@pytest.mark.parametrize("Mr,K,N,gs,zeros,act", [
    (512, 4096, 1032, 128, True, True),   # ragged last column block
    (200, 2048, 776, 64, False, False),
    (129, 1024, 520, 256, True, False),
])
def test_gemm_tile_widths_agree(gpu, orc, Mr, K, N, gs, zeros, act, tune):
    """128 x 128 workgroup tiles (one 32-column block per wave, chosen for
    small grids) and 128 x 256 tiles give the same C bit for bit (same k
    order per output) and meet the oracle's bar."""
    c = orc.gptq_case(90 + gs, K, N, gs, zeros=zeros, act_order=act, M=Mr, x_dtype=np.float16)
    w = up(gpu, c)
    ys = {}
    for cb in ("1", "2"):
        tune(GEMM_CB=int(cb))
        tune(GEMM_NO_SPLIT=1)
        ys[cb] = run_gemm(gpu, w, c["x"])
    ref = orc.gptq_matvec_f64(c["x"], c["qweight"], c["scales"], K, N, gs, qzeros=c["qzeros"], g_idx=c["g_idx"])
    assert np.array_equal(ys["1"], ys["2"])
    assert orc.rel_l2(ys["1"], ref) < 5e-4


def test_gemm_long_k(gpu, orc, route):
    Mr, K, N, gs = 80, 32768, 264, 128
    c = orc.gptq_case(120, K, N, gs, zeros=True, act_order=True, M=Mr, x_dtype=np.float16)
    w = up(gpu, c)
    y = run_gemm(gpu, w, c["x"])
    ref = orc.gptq_matvec_f64(c["x"], c["qweight"], c["scales"], K, N, gs, qzeros=c["qzeros"], g_idx=c["g_idx"])
    assert orc.rel_l2(y, ref) < 5e-4


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.float16])
def test_gemm_unaligned_c_matches_aligned(gpu, orc, out_dtype, route):
    """C one element past a 16-byte boundary takes the GEMM's per-element
    epilogue, an aligned C the one staged through LDS (16-byte row chunks; K
    too short to be split, whose partials are aligned): the same values bit
    for bit. The skinny kernel writes elements either way."""
    Mr, K, N, gs = 130, 512, 264, 128
    c = orc.gptq_case(77, K, N, gs, zeros=True, M=Mr, x_dtype=np.float16)
    w = up(gpu, c)
    a = torch.from_numpy(c["x"]).to(gpu.device)
    aligned = torch.empty(Mr, N, dtype=out_dtype, device=gpu.device)
    base = torch.empty(Mr * N + 1, dtype=out_dtype, device=gpu.device)
    shifted = base[1:].view(Mr, N)
    assert shifted.data_ptr() % 16 != 0
    for cc in (aligned, shifted):
        M.gptq_gemm(gpu, a, w.qweight, w.scales, cc, K, N, gs, w.qzeros, w.perm, w.flags)
    torch.cuda.synchronize()
    assert torch.equal(aligned, shifted)
    ref = orc.gptq_matvec_f64(c["x"], c["qweight"], c["scales"], K, N, gs, qzeros=c["qzeros"])
    assert orc.rel_l2(aligned.float().cpu().numpy(), ref) < 5e-4


def run_gate_up(gpu, wg, wu, a_np, out_dtype=torch.float32):
    a = torch.from_numpy(np.ascontiguousarray(a_np, dtype=np.float16)).to(gpu.device)
    cg = torch.full((a.shape[0], wg.N), float("nan"), dtype=out_dtype, device=gpu.device)
    cu = torch.full_like(cg, float("nan"))
    M.gate_up_gemm(gpu, a, wg.qweight, wg.scales, wu.qweight, wu.scales, cg, cu, wg.K, wg.N, wg.group_size,
                   wg.qzeros, wu.qzeros, wg.perm, wg.flags)
    torch.cuda.synchronize()
    return cg.float().cpu().numpy(), cu.float().cpu().numpy()


@pytest.mark.parametrize("Mr,K,N,gs,zeros,act,tiled,out", [
    (512, 2560, 9728, 128, False, False, True, torch.float16),  # configs[4] gate/up at a 512-token prefill: one grid
    (300, 1536, 776, 64, True, True, False, torch.float32),     # act-order, zeros, row-major qweight
    (257, 2048, 520, 256, True, False, True, torch.float16),    # group 256, ragged M
    (64, 4096, 264, 128, False, False, True, torch.float32),    # few tiles: split-K, two launches on one A
    (300, 4096, 264, 128, False, False, True, torch.float32),   # the same beyond the skinny kernel's rows
    (33, 1024, 1032, 128, "up", False, True, torch.float32),    # zero points on up only
    (128, 2560, 9728, 128, False, False, True, torch.float16),  # a short prompt: the skinny kernel, one launch per weight
])
def test_gate_up_gemm_equals_two_gemms(gpu, orc, Mr, K, N, gs, zeros, act, tiled, out):
    """st_gptq_i4_gate_up_gemm: each output bit for bit what st_gptq_i4_gemm
    gives for that weight (one grid over both weights' tiles, or two
    launches on the shared pre-processed A when K is split, or the skinny
    kernel once per weight), and within the GEMM bar of the f64 oracle."""
    cg = orc.gptq_case(600 + Mr, K, N, gs, zeros=zeros is True, act_order=act, M=Mr, x_dtype=np.float16)
    cu = orc.gptq_case(700 + Mr, K, N, gs, zeros=bool(zeros), act_order=act)
    cu["g_idx"] = cg["g_idx"]
    wg, wu = up(gpu, cg, tiled=tiled), up(gpu, cu, tiled=tiled)
    assert (wg.qzeros is None) == (zeros is not True) and (wu.qzeros is None) == (not zeros)
    yg, yu = run_gate_up(gpu, wg, wu, cg["x"], out)
    np.testing.assert_array_equal(yg, run_gemm(gpu, wg, cg["x"], out))
    np.testing.assert_array_equal(yu, run_gemm(gpu, wu, cg["x"], out))
    for cc, y in ((cg, yg), (cu, yu)):
        ref = orc.gptq_matvec_f64(cg["x"], cc["qweight"], cc["scales"], K, N, gs, qzeros=cc["qzeros"],
                                  g_idx=cg["g_idx"])
        e = orc.rel_l2(y, ref)
        print(f"gate/up gemm M={Mr} K={K} N={N} gs={gs} zeros={zeros} act={act}: rel-L2 {e:.3e}")
        assert e < TOL


def test_gate_up_gemm_graph_replay(gpu, orc, route):
    """Captured once, replayed three times with eager work between: both
    outputs equal the eager call's bit for bit every time."""
    Mr, K, N, gs = 256, 1024, 2048, 128
    cg = orc.gptq_case(80, K, N, gs, zeros=True, M=Mr, x_dtype=np.float16)
    cu = orc.gptq_case(81, K, N, gs, zeros=True)
    wg, wu = up(gpu, cg), up(gpu, cu)
    a = torch.from_numpy(cg["x"].astype(np.float16)).to(gpu.device)
    eg, eu = (torch.empty(Mr, N, device=gpu.device) for _ in range(2))
    call = lambda g_, u_: M.gate_up_gemm(gpu, a, wg.qweight, wg.scales, wu.qweight, wu.scales, g_, u_, K, N, gs,
                                         wg.qzeros, wu.qzeros, None, wg.flags)
    call(eg, eu)
    torch.cuda.synchronize()
    og, ou = torch.empty_like(eg), torch.empty_like(eu)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        call(og, ou)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            call(og, ou)
    for i in range(3):
        og.fill_(float("nan"))
        ou.fill_(float("nan"))
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(og, eg) and torch.equal(ou, eu), f"replay {i}"
        call(eg, eu)  # eager work between
        torch.cuda.synchronize()


@pytest.mark.parametrize("Mr,K,N,gs,act,pair", [
    (64, 1024, 9000, 128, False, "i4xs_kernel"),     # up to 64 tokens: the skinny kernel
    (77, 2560, 9728, 128, False, "i4xs_kernel"),
    (124, 4864, 11248, 256, False, "gemm_kernel"),   # the GEMM's grid of both weights is the faster one
    (139, 4608, 11968, 128, True, "gemm_kernel"),
    (150, 4608, 1048, 64, True, "i4xs_kernel"),      # weights that narrow: by one alone
    (256, 1024, 1032, 128, False, "i4xs_kernel"),
    (161, 5120, 5952, 128, False, "gemm_kernel"),    # above 160 tokens and 2^24 values
    (257, 1024, 1032, 128, False, "gemm_kernel"),
])
def test_gate_up_takes_the_kernel_of_single_calls(gpu, Mr, K, N, gs, act, pair):
    """One rule for both kinds of call, on both sides of its lines: a gate/up
    call takes the kernel of a single call, and gives its bits."""
    g = torch.Generator(device="cuda").manual_seed(Mr)
    qw = [torch.randint(-2**31, 2**31, (sta.lib().st_gptq_i4_tiled_words(K, N, gs),), dtype=torch.int32, device="cuda", generator=g)
          for _ in range(2)]
    sc = [(torch.rand(K // gs, N, device="cuda", generator=g) * 0.01).half() for _ in range(2)]
    qz = torch.randint(-2**31, 2**31, (K // gs, N // 8), dtype=torch.int32, device="cuda", generator=g)  # (up's: gate has none)
    perm = torch.randperm(K, device="cuda", generator=g).int() if act else None
    a = torch.randn(Mr, K, device="cuda", generator=g).half()
    y = [torch.full((Mr, N), float("nan"), device="cuda") for _ in range(4)]
    launches()
    M.gate_up_gemm(gpu, a, qw[0], sc[0], qw[1], sc[1], y[0], y[1], K, N, gs, up_qz=qz, perm=perm, flags=2)
    ran = launches()
    for i in range(2):
        M.gptq_gemm(gpu, a, qw[i], sc[i], y[2 + i], K, N, gs, (None, qz)[i], perm, 2)
    torch.cuda.synchronize()
    assert {"gemm_kernel", "i4xs_kernel"} & set(ran) == {pair} == {"gemm_kernel", "i4xs_kernel"} & set(launches())
    assert torch.equal(y[0], y[2]) and torch.equal(y[1], y[3])


@pytest.mark.parametrize("out", [torch.float32, torch.float16])
@pytest.mark.parametrize("Mr,K,N,gs", [(300, 4096, 264, 128), (129, 8192, 1032, 64), (700, 2048, 136, 256)])
def test_gate_up_gemm_splits_in_one_grid(gpu, orc, Mr, K, N, gs, out, tune):
    """Where a single call splits K, both weights' splits are one grid and one
    reduction, of which either weight's half is a single call's."""
    tune(GEMM_CB=0)
    cg = orc.gptq_case(800 + Mr, K, N, gs, zeros=True, M=Mr, x_dtype=np.float16)
    cu = orc.gptq_case(900 + Mr, K, N, gs)
    wg, wu = up(gpu, cg), up(gpu, cu)
    launches()
    yg, yu = run_gate_up(gpu, wg, wu, cg["x"], out)
    assert launches() == ["prep_a_kernel", "gemm_kernel", "splitk_reduce_kernel"]
    np.testing.assert_array_equal(yg, run_gemm(gpu, wg, cg["x"], out))
    np.testing.assert_array_equal(yu, run_gemm(gpu, wu, cg["x"], out))
    assert "splitk_reduce_kernel" in launches()
    assert orc.rel_l2(yu, orc.gptq_matvec_f64(cg["x"], cu["qweight"], cu["scales"], K, N, gs)) < 5e-4
