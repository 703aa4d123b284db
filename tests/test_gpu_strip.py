"""The strip kernel (q4_strip.hip: fp32 activations, at most 512 columns, one
round of blocks) at its two block heights, short last row blocks, one and
several column blocks with ragged ends, one round of K and several, every
group size, either side of its limits, against the fp64 oracle on the cast
activations (cast_f32_to_f16, Kernels.swift:816-822; DiTLinear.applyF32in's q4
branch, DiTModel.swift:102-125) and, where its grid ends, against the GEMM."""
import numpy as np
import pytest

from helpers import TOL_GEMM_F16, assert_parity, host, plan
from oracle import q4_oracle as o

pytestmark = pytest.mark.gpu


# (M, N, K, g, rows of a block; 0: past the kernel's limits, the GEMM).  32-row
# blocks up to 8192 / ceil(N / 128) rows, then 64-row ones up to twice that; K %
# 128 == 0 and at most 64 groups; K > 2048 from M N = 2^18.
SHAPES = [(1, 128, 128, 64, 32), (31, 1, 256, 32, 32), (33, 130, 2048, 32, 32), (777, 127, 1152, 128, 32),
          (6144, 128, 2048, 64, 32), (8192, 100, 128, 64, 32), (8193, 100, 128, 64, 64),
          (4096, 256, 2048, 32, 32), (4097, 256, 2048, 32, 64), (2731, 384, 384, 128, 64),
          (2700, 512, 640, 64, 64), (16384, 65, 128, 128, 64), (16385, 65, 128, 128, 0),
          (4096, 512, 2048, 64, 64), (4097, 512, 2048, 64, 0), (2048, 128, 4096, 64, 32),
          (2047, 128, 4096, 64, 0), (600, 500, 3072, 128, 32), (500, 500, 4096, 64, 0),
          (600, 500, 4224, 128, 0), (600, 500, 2176, 32, 0), (100, 128, 2080, 32, 0)]


@pytest.mark.parametrize("M,N,K,g,block", SHAPES)
def test_strip(pkg, dev, M, N, K, g, block):
    import torch
    got = plan(pkg, M, N, K, g, x_dtype=torch.float32)
    assert got.route == "gemm" and (got.rows == block if block else got.rows >= 128)
    gen = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=gen, device=dev)
    x[M // 2, K // 3] = 1e6          # clamped
    x[M - 1, 5] = float("-inf")
    x[0, 7] = float("nan")           # the lower bound
    w = torch.randint(-2**31, 2**31 - 1, (N, K // 8), generator=gen, device=dev, dtype=torch.int64).int()
    s = (torch.randn(N, K // g, generator=gen, device=dev) * 0.02).abs().half()
    W = pkg.Q4Weight(w, s, s * -8.0, K, g)
    bias = torch.randn(N, generator=gen, device=dev)
    y = pkg.matmul_q4_ex(x, W, M, N, out_dtype=torch.float32)
    yb = pkg.matmul_q4_ex(x, W, M, N, out_dtype=torch.float32, bias=bias,
                          epilogue=pkg.SLTX_EPI_GELU_TANH)
    yh = pkg.matmul_q4_ex(x, W, M, N, out_dtype=torch.bfloat16)
    torch.cuda.synchronize()
    assert torch.equal(yh, y.bfloat16())
    rows = np.unique(np.clip([0, 1, 31, 32, 63, 64, M // 2, M - 33, M - 2, M - 1], 0, M - 1))
    x16 = o.cast_f32_to_f16_ref(host(x)[rows])
    ref = o.matmul_q4_f64(x16, host(w), host(s), host(W.biases), g)
    got = y.cpu().numpy()[rows]
    clamped = np.abs(x16.astype(np.float64)).max(1) > 6e4
    for sel, what in ((clamped, "clamped rows"), (~clamped, "other rows")):
        if sel.any():
            assert_parity(got[sel], ref[sel], TOL_GEMM_F16, f"M={M} N={N} K={K} g={g} {what}")
    # the epilogue on the same sums: fp32 gelu of values at most 1e-6 off
    want = o.gelu_tanh_f64(got.astype(np.float64) + host(bias))
    assert np.abs(yb.cpu().numpy()[rows] - want).max() <= 1e-5 * (1 + np.abs(want).max())


def test_strip_graph(pkg, dev):
    """Captured without an eager call before (no workspace is needed), replayed
    with other work between: every replay equals the eager result bit for bit."""
    import torch
    M, N, K, g = 500, 200, 1024, 64
    gen = torch.Generator(device=dev).manual_seed(1)
    x = torch.randn(M, K, generator=gen, device=dev)
    w = torch.randint(-2**31, 2**31 - 1, (N, K // 8), generator=gen, device=dev, dtype=torch.int64).int()
    s = (torch.randn(N, K // g, generator=gen, device=dev) * 0.02).abs().half()
    W = pkg.Q4Weight(w, s, s * -8.0, K, g)
    want = pkg.matmul_q4_ex(x, W, M, N)
    out = torch.empty_like(want)
    torch.cuda.synchronize()
    st = torch.cuda.Stream()
    gr = torch.cuda.CUDAGraph()
    with torch.cuda.graph(gr, stream=st):
        pkg.matmul_q4_ex(x, W, M, N, out=out, stream=st)
    for _ in range(3):
        out.zero_()
        pkg.matmul_q4_ex(x, W, M, N)
        torch.cuda.synchronize()
        gr.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
