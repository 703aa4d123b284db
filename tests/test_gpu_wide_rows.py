"""The wide-M route beyond 256 rows and beyond 64 scale groups per block
(q4_wide.hip): one to 48 blocks along M of 33-128 rows, the last one short,
K of one round up to 4096 with a full 128-group slab at group 32, ragged N,
and either side of its limits (K per block, X bytes, one round of blocks),
against the fp64 oracle on rows at the block edges.  Same semantics as every
M > 1 route (matmulQ4Fast / matmulQ4FastF32, Ops.swift:312-381)."""
import numpy as np
import pytest
import torch   # before the library: both then use torch's HIP runtime

from helpers import GATE, TOL_GEMM_F16, assert_parity, gpu_inputs, host, rounded_weights_f16
from oracle import q4_oracle as o

SHAPES = [(257, 3072, 3072, 64), (333, 3072, 3072, 32), (385, 1000, 4096, 32), (640, 3072, 2048, 64),
          (1000, 2048, 2048, 128), (300, 777, 1280, 64), (700, 65, 128, 32), (6143, 128, 2048, 64),
          (129, 1025, 4096, 32), (100, 2048, 8192, 128)]
PAIRS = [(96, 2000, 3072, 32), (70, 100, 4096, 32), (300, 333, 1024, 128)]


def _rows(M):
    return np.unique(np.clip([0, 1, 31, 32, 63, 64, 95, 96, 127, 128, M // 2, M - 33, M - 2, M - 1], 0, M - 1))


@pytest.mark.parametrize("M,N,K,g", SHAPES)
def test_shapes_run_the_wide_route(pkg, M, N, K, g):
    assert pkg.gemm_route(M, N, K, group_size=g) == "wide"


def test_limits(pkg):
    assert all(pkg.gemm_route(*s[:3], group_size=s[3], gated=True) == "wide" for s in PAIRS)
    assert pkg.gemm_route(640, 3072, 3072) == "wide" and pkg.gemm_route(641, 3072, 3072) == "gemm"   # one round
    assert pkg.gemm_route(300, 3072, 8192) == "gemm"                                                 # K per block
    assert pkg.gemm_route(8192, 64, 2048) == "wide" and pkg.gemm_route(8193, 64, 2048) == "gemm"     # X bytes


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,g", SHAPES)
def test_rows(pkg, dev, M, N, K, g):
    x, [(w, s, b)] = gpu_inputs(M, N, K, g, seed=M + N, dev=dev)
    y32 = pkg.matmul_q4_fast_f32(x, w, s, b, M, K, N, g)
    y16 = pkg.matmul_q4_fast(x, w, s, b, M, K, N, g)
    gen = torch.Generator(device=dev).manual_seed(M)
    res = torch.randn(M, N, generator=gen, device=dev).half()
    bias = torch.randn(N, generator=gen, device=dev)
    W = pkg.Q4Weight(w, s, b, K, g)
    yr = pkg.matmul_q4_residual(x, W, res, M, N)
    yb = pkg.matmul_q4_ex(x, W, M, N, bias=bias, epilogue=pkg.SLTX_EPI_GELU_TANH)
    torch.cuda.synchronize()
    assert torch.equal(y16, y32.half())
    assert torch.equal(yr, (res.float() + y16.float()).half())
    rows = _rows(M)
    ref = o.matmul_q4_f64(host(x)[rows].astype(np.float64), host(w), host(s), host(b), g)
    assert_parity(y32.cpu().numpy()[rows], ref, TOL_GEMM_F16, f"M={M} N={N} K={K} g={g}")
    # the epilogue on the same fp32 sums: fp32 gelu of a value 1e-6 off at most
    want = o.gelu_tanh_f64(y32.cpu().numpy()[rows].astype(np.float64) + host(bias))
    got = yb.cpu().numpy()[rows]
    assert np.abs(got - want).max() <= 1e-5 * (1 + np.abs(want).max())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,g", PAIRS)
def test_pairs(pkg, dev, M, N, K, g):
    x, sets = gpu_inputs(M, N, K, g, seed=K, dev=dev, n_weights=2)
    y = pkg.matmul_q4_silu_mul(x, *(pkg.Q4Weight(*t, K, g) for t in sets), M, K, N)
    torch.cuda.synchronize()
    rows = _rows(M)
    xs = host(x)[rows].astype(np.float64)
    got = y.cpu().numpy()[rows].astype(np.float64)
    (wg, sg, bg), (wu, su, bu) = (tuple(host(t) for t in st) for st in sets)
    ref = o.silu_mul_f64(o.matmul_q4_f64(xs, wg, sg, bg, g), o.matmul_q4_f64(xs, wu, su, bu, g))
    assert o.max_rel_err(got, ref) <= GATE
    # elementwise on the fp16-rounded weights: fp32 sums, exp2 / rcp, one fp16 rounding
    ref_w = o.silu_mul_f64(xs @ rounded_weights_f16(wg, sg, bg, g).T, xs @ rounded_weights_f16(wu, su, bu, g).T)
    ok, worst = o.elementwise_ok(got, ref_w, rtol=1e-3, atol_rms=1e-4)
    assert ok, f"{worst:.2f}x the allowance"
