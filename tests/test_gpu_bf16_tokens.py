"""The bf16 matvec of 2-8 tokens (bf16mm_kernel: matrix cores, x as two or
three bf16 parts) at the edges of its row groups, segments and LDS, with
infinities, NaNs and values whose parts leave bf16's range."""
import numpy as np
import pytest
import torch

from shady_thinker_amd import model as M

pytestmark = pytest.mark.gpu

# Exact products; what is left are K / 256 + 8 roundings of f32 sums, of both
# signs: sqrt(28) 2^-23 = 6.3e-7 at K = 5120.
TOL = 6.5e-7


def _run(gpu, x, w):
    y = torch.full((x.shape[0], w.shape[0]), 7.0, device="cuda")
    M.bf16_matvec(gpu, x, w, y, w.shape[1], w.shape[0])
    torch.cuda.synchronize()
    return y.cpu()


def _case(seed, K, N, Mr):
    g = torch.Generator().manual_seed(seed)
    x, w = torch.randn(Mr, K, generator=g), torch.randn(N, K, generator=g).to(torch.bfloat16)
    x[:, torch.randint(0, K, (max(1, K // 256),), generator=g)] *= 16.0
    return x, w


@pytest.mark.parametrize("K,N,Mr,f16", [
    (8, 1, 2, False),        # one piece of a segment, one row
    (64, 9, 8, False),
    (72, 1001, 5, True),     # a second segment of one piece, ragged rows
    (320, 2049, 3, False),   # five segments: a batch and one
    (1000, 4099, 7, False),  # more groups than waves of one per CU
    (2560, 33000, 4, True),  # several groups per wave
    (5120, 264, 8, False),   # x fills the LDS
    (10232, 100, 3, False),
])
def test_bf16_tokens(gpu, K, N, Mr, f16):
    x, w = _case(K + N, K, N, Mr)
    x = x.half() if f16 else x
    y = _run(gpu, x.cuda(), w.cuda()).double()
    ref = x.double() @ w.double().t()
    assert ((y - ref).norm() / ref.norm()).item() < TOL


def test_bf16_tokens_nonfinite(gpu):
    """Infinities and NaNs of x and of weights give what f32 sums give."""
    K, N, Mr = 520, 70, 6
    x, w = _case(5, K, N, Mr)
    x[1, 3], x[2, 100], x[2, 101], x[4, 519] = float("inf"), float("-inf"), float("inf"), float("nan")
    w[5, 7], w[6, 9], w[69, 500] = float("inf"), float("nan"), float("-inf")
    y = _run(gpu, x.cuda(), w.cuda()).numpy()
    ref = (x @ w.float().t()).numpy()
    assert np.array_equal(np.isnan(y), np.isnan(ref))
    assert np.array_equal(y[np.isinf(ref)], ref[np.isinf(ref)]) and np.isinf(y).sum() == np.isinf(ref).sum()
    ok = np.isfinite(ref)
    assert np.allclose(y[ok], ref[ok], rtol=1e-4, atol=1e-3)


def test_bf16_tokens_scales_of_x(gpu):
    """Rows of very different size, down to where the parts of x fall below
    bf16's range, a zero row and f32 subnormals: each row by itself."""
    K, N, Mr = 1024, 264, 8
    x, w = _case(6, K, N, Mr)
    scale = torch.tensor([1e30, 1e10, 1.0, 1e-10, 1e-25, 1e-34, 1e-36, 0.0])
    x = x * scale[:, None]
    y = _run(gpu, x.cuda(), w.cuda()).double()
    ref = x.double() @ w.double().t()
    assert not y[7].any()
    for r in range(7):
        assert ((y[r] - ref[r]).norm() / ref[r].norm()).item() < TOL, r


@pytest.mark.parametrize("xs,ws", [
    (2.0**-120, 2.0**50),   # x's third part below 2^-133
    (2.0**-140, 2.0**60),   # x below f32's normals
    (2.0**60, 2.0**-130),   # weights below bf16's normals
    (2.0**-20, 2.0**-110),  # sums below f32's normals
    (2.0**110, 2.0**-20),   # x past the staging scale's range
])
def test_bf16_tokens_far_scales(gpu, xs, ws):
    """Small x against large weights and the other way: no part of x is lost
    whatever the size of the sum."""
    K, N, Mr = 1000, 264, 5
    x, w = _case(7, K, N, Mr)
    x, w = x * xs, (w.float() * ws).to(torch.bfloat16)
    y = _run(gpu, x.cuda(), w.cuda()).double()
    ref = x.double() @ w.double().t()
    tiny = ref.abs().max() < 2.0**-120  # f32's steps below its normals
    assert ((y - ref).norm() / ref.norm()).item() < (2.0**-149 * (K * N * Mr) ** 0.5 / ref.norm().item() + TOL if tiny else TOL)


def test_bf16_tokens_one_bad_token(gpu):
    """A NaN and an infinity in two tokens of a call over many rows: theirs are
    what f32 sums give, the other tokens' are bit for bit what they are without."""
    K, N, Mr = 520, 20001, 8
    x, w = _case(8, K, N, Mr)
    good = _run(gpu, x.cuda(), w.cuda())
    x[2, 7], x[6, 500] = float("nan"), float("inf")
    y = _run(gpu, x.cuda(), w.cuda())
    keep = [0, 1, 3, 4, 5, 7]
    assert torch.equal(y[keep], good[keep]) and torch.isnan(y[2]).all()
    ref = x[6] @ w.float().t()
    assert torch.equal(torch.isnan(y[6]), torch.isnan(ref)) and torch.equal(y[6][torch.isinf(ref)], ref[torch.isinf(ref)])
