"""The prefill GEMM's workgroup tiles (128 x 128, 128 x 256 and 128 x 512,
GEMM_CB 1..3): the same C bit for bit from each (the same k order per
output), ragged rows and columns, f32 and f16 C, GPTQ and INT8, against the
f64 oracle; and the split that the launcher chooses itself."""
import numpy as np
import pytest
import torch

import shady_thinker_amd as sta
from shady_thinker_amd import model as M

pytestmark = pytest.mark.gpu

TOL = 3e-4  # one f16 rounding per weight: 2^-11 / sqrt(3) rms at worst
TOL_I8 = 1e-6  # exact products, f32 sums


@pytest.mark.parametrize("Mr,K,N,gs,zeros,out", [
    (129, 384, 520, 128, True, torch.float32),    # three K tiles, one column block past 512
    (300, 1024, 1032, 64, False, torch.float16),
    (257, 1280, 504, 256, True, torch.float32),   # less than one 512-column tile
    (128, 128, 2056, 128, False, torch.float16),  # one K tile
])
def test_gemm_tiles_agree(gpu, orc, Mr, K, N, gs, zeros, out, tune):
    c = orc.gptq_case(1200 + Mr, K, N, gs, zeros=zeros, M=Mr, x_dtype=np.float16)
    w = sta.GptqWeight.upload(gpu, c["qweight"], c["scales"], gs, qzeros=c["qzeros"])
    a = torch.from_numpy(c["x"]).cuda()
    ys = []
    for cb in (1, 2, 3):
        tune(GEMM_CB=cb, GEMM_NO_SPLIT=1)
        y = torch.full((Mr, N), float("nan"), device="cuda", dtype=out)
        M.gptq_gemm(gpu, a, w.qweight, w.scales, y, K, N, gs, w.qzeros, None, w.flags)
        torch.cuda.synchronize()
        ys.append(y)
    assert torch.equal(ys[0], ys[1]) and torch.equal(ys[0], ys[2])
    ref = orc.gptq_matvec_f64(c["x"], c["qweight"], c["scales"], K, N, gs, qzeros=c["qzeros"])
    assert orc.rel_l2(ys[0].float().cpu().numpy(), ref) < TOL * (2**0.5 if out == torch.float16 else 1)


@pytest.mark.parametrize("Mr,K,N,tiled,cbs", [
    (129, 384, 516, True, (1, 2, 3)),
    (300, 640, 1028, False, (1, 2, 3)),
    (64, 5120, 1300, True, (0,)),  # the launcher's own choice: K split
])
def test_int8_gemm_tiles_agree(gpu, orc, Mr, K, N, tiled, cbs, tune):
    c = orc.int8_case(1300 + Mr, K, N, M=Mr)
    x = c["x"].astype(np.float16)
    w = sta.Int8Weight.upload(gpu, c["w"], c["scale"], tiled=tiled)
    a = torch.from_numpy(x).cuda()
    ys = []
    for cb in cbs:
        if cb:
            tune(GEMM_CB=cb, GEMM_NO_SPLIT=1)
        y = torch.full((Mr, N), float("nan"), device="cuda")
        M.int8_gemm(gpu, a, w.w, w.scale, y, K, N, w.flags)
        torch.cuda.synchronize()
        ys.append(y)
    assert all(torch.equal(ys[0], y) for y in ys)
    assert orc.rel_l2(ys[0].cpu().numpy(), orc.int8_matvec_f64(x, c["w"], c["scale"], K, N)) < TOL_I8
