"""sltx_matmul_q4_residual_rms_norm at the row counts where it runs a route
other than the GEMM (narrow, small-M, mid-M with and without K halves, wide
with and without K splits, the two-row GEMV): it equals the unfused sequence
of the same library bit for bit (linear + residualRmsNorm, Ops.swift:256-279;
linear + elemAdd + rmsNorm, LlamaModel.swift:278-279, 233), and the GEMM on
either side of the last routed M; also in place on the residual stream."""
import pytest

from helpers import gpu_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K,g", [(3072, 3072, 64), (3072, 8192, 32), (1000, 4096, 128)])
@pytest.mark.parametrize("M", [1, 2, 3, 8, 17, 32, 33, 100, 256, 257])
def test_equals_unfused(pkg, dev, M, N, K, g):
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
    want_n2 = pkg.rms_norm(want_r, nw, 1e-5, M, N)
    inplace = res.clone()
    got_r2, got_n2 = pkg.matmul_q4_residual_rms_norm(x, W, inplace, nw, 1e-5, M, N, True,
                                                     residual_out=inplace)
    torch.cuda.synchronize()
    if pkg.gemm_route(M, N, K, g) != "gemm":
        assert torch.equal(got_r, want_r) and torch.equal(got_n, want_n)
        assert torch.equal(got_r2, want_r) and torch.equal(got_n2, want_n2)
    else:   # its split count may differ from the unfused call's: one fp16 rounding
        for a, c in ((got_r, want_r), (got_n, want_n), (got_r2, want_r), (got_n2, want_n2)):
            assert float((a.float() - c.float()).norm() / c.float().norm()) < 2.0**-11
