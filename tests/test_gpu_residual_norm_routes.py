"""sltx_matmul_q4_residual_rms_norm on every route -- narrow, small-M, mid-M with
and without K halves, wide with and without K splits, the two-row GEMV, the GEMM
unsplit and, in the pass that adds its partial sums, at every split count and row
length that pass is compiled for -- equals the unfused sequence of the same
library bit for bit (linear + residualRmsNorm, Ops.swift:256-279; linear +
elemAdd + rmsNorm, LlamaModel.swift:278-279, 233); also in place on the residual
stream."""
import pytest

from helpers import gpu_inputs, plan

pytestmark = pytest.mark.gpu


# (M, N, K, g, splits): 256-thread rows of one, two, up to four and up to eight
# 8-wide pieces (N <= 2048, 4096, 8192, 16384) by 2, 3, 4 and more splits
SPLIT = [
    (800, 1800, 4224, 64, 2), (1200, 1000, 4352, 128, 3), (1500, 520, 4224, 32, 4), (700, 1000, 4224, 64, 5),
    (700, 2056, 4352, 128, 2), (900, 2056, 3072, 64, 3), (257, 2560, 4224, 32, 4), (257, 2056, 4224, 64, 5),
    (257, 3072, 8192, 64, 7), (257, 4096, 16384, 64, 8),
    (257, 5120, 4224, 64, 2), (400, 4104, 3072, 32, 3), (257, 5120, 5120, 64, 4), (257, 4104, 4224, 64, 5),
    (400, 8200, 4096, 128, 2), (600, 8200, 10240, 64, 3), (400, 12288, 16384, 64, 4), (257, 8200, 16384, 64, 5),
    # the generic GEMM (K % 128 != 0)
    (300, 2048, 4160, 64, 7),
]


@pytest.mark.parametrize("N,K,g", [(3072, 3072, 64), (3072, 8192, 32), (1000, 4096, 128)])
@pytest.mark.parametrize("M", [1, 2, 3, 8, 17, 32, 33, 100, 256, 257])
def test_equals_unfused(pkg, dev, M, N, K, g):
    _equals_unfused(pkg, dev, M, N, K, g)


@pytest.mark.parametrize("M,N,K,g,splits", SPLIT)
def test_split_gemm_equals_unfused(pkg, dev, M, N, K, g, splits):
    assert plan(pkg, M, N, K, g)[:2] == ("gemm", splits)
    _equals_unfused(pkg, dev, M, N, K, g)


def _equals_unfused(pkg, dev, M, N, K, g):
    import torch
    x, [(w, s, b)] = gpu_inputs(M, N, K, g, seed=M + N, dev=dev)
    gen = torch.Generator(device=dev).manual_seed(M)
    res = torch.randn(M, N, generator=gen, device=dev).half()
    nw = 1.0 + 0.1 * torch.randn(N, generator=gen, device=dev)
    W = pkg.Q4Weight(w, s, b, K, g)
    o = pkg.matmul_q4_fast(x, w, s, b, M, K, N, g)
    want_r, want_n = pkg.residual_rms_norm(res, o, nw, 1e-5, M, N)
    got_r, got_n = pkg.matmul_q4_residual_rms_norm(x, W, res, nw, 1e-5, M, N, False)
    # the stored sum is the same for both variants; its norm is of the rounded sum
    # (unfused: the residual epilogue, at M = 1 the GEMV's)
    want_r2 = pkg.matmul_q4_residual(x, W, res, M, N) if M > 1 else want_r
    want_n2 = pkg.rms_norm(want_r2, nw, 1e-5, M, N)
    inplace = res.clone()
    got_r2, got_n2 = pkg.matmul_q4_residual_rms_norm(x, W, inplace, nw, 1e-5, M, N, True,
                                                     residual_out=inplace)
    torch.cuda.synchronize()
    assert torch.equal(got_r, want_r) and torch.equal(got_n, want_n)
    assert torch.equal(got_r2, want_r2) and torch.equal(got_r2, want_r) and torch.equal(got_n2, want_n2)
