"""Where the small-M route takes X from (q4_skinny.hip): at most 8 rows, one
load filling two fragments, or LDS; 9..16 rows through LDS or registers.

The same K slices, steps and order of addition run in each, so the first 8 of
M > 8 rows must equal those 8 rows alone bit for bit, for every step count of
8 and 16 waves.  K = 12288 and 14336 (16 waves of 6 and 7 steps) run only at
M <= 8 and are checked against the fp64 oracle with the GEMM's tolerance."""
import numpy as np
import pytest

from helpers import TOL_GEMM_F16, assert_parity, gpu_inputs, host, plan, q4w, to_dev
from oracle import q4_oracle as o

pytestmark = pytest.mark.gpu


# (M of the larger call, N, K, g)
SAME = [(16, 33, 1024, 32), (16, 100, 2048, 64), (9, 48, 3072, 64), (16, 100, 3072, 128),
        (15, 40, 4096, 32), (16, 40, 4096, 64), (16, 33, 5120, 64), (16, 20, 6144, 64),
        (12, 40, 8192, 64), (12, 4200, 10240, 64)]


@pytest.mark.parametrize("M,N,K,g", SAME)
def test_rows_alone_and_among_more(pkg, dev, M, N, K, g):
    import torch
    assert pkg.gemm_route(M, N, K, group_size=g) == "small_m"
    x, [(w, s, b)] = o.make_inputs(M, N, K, g, seed=M + N + K)
    tx, args = to_dev(x, dev), [to_dev(a, dev) for a in (w, s, b)]
    want = pkg.matmul_q4_fast_f32(tx, *args, M, K, N, g)
    for m in (5, 8):
        assert pkg.gemm_route(m, N, K, group_size=g) == "small_m"
        y = pkg.matmul_q4_fast_f32(tx[:m].contiguous(), *args, m, K, N, g)
        assert torch.equal(y, want[:m]), m


@pytest.mark.parametrize("M,N,K", [(16, 72, 2048), (16, 40, 3072), (16, 4200, 3072), (16, 40, 8192)])
def test_pair_rows_alone_and_among_more(pkg, dev, M, N, K):
    import torch
    g = 64
    x, ws = o.make_inputs(M, N, K, g, seed=N + K, n_weights=2)
    gate, up = [q4w(pkg, *w, K, g, dev) for w in ws]
    tx = to_dev(x, dev)
    assert pkg.gemm_route(M, N, K, gated=True) == "small_m"
    want = pkg.matmul_q4_silu_mul(tx, gate, up, M, K, N)
    for m in (2, 3, 8):   # (one row takes the GEMV)
        y = pkg.matmul_q4_silu_mul(tx[:m].contiguous(), gate, up, m, K, N)
        assert torch.equal(y, want[:m]), m


@pytest.mark.parametrize("g", [32, 64, 128])
@pytest.mark.parametrize("K", [2048, 3072])
@pytest.mark.parametrize("M", [5, 6, 7, 8])
def test_few_rows_in_lds_equal_halves(pkg, dev, M, K, g):
    """4200 weight rows take X from LDS, 4000 (one block per CU) as halves."""
    import torch
    x, [(w, s, b)] = gpu_inputs(M, 4200, K, g, seed=M + K, dev=dev)
    assert [plan(pkg, M, N, K, g)[0::2] for N in (4200, 4000)] == [("small_m", 1), ("small_m", 2)]
    y = pkg.matmul_q4_fast_f32(x, w, s, b, M, K, 4200, g)
    part = pkg.matmul_q4_fast_f32(x, w[:4000], s[:4000], b[:4000], M, K, 4000, g)
    torch.cuda.synchronize()
    assert torch.equal(y[:, :4000], part)
    assert_parity(y.cpu().numpy(), o.matmul_q4_f64(host(x).astype(np.float64), host(w), host(s), host(b), g),
                  TOL_GEMM_F16, f"M={M} K={K} g={g}")


@pytest.mark.parametrize("K,g", [(12288, 32), (12288, 128), (14336, 64), (14336, 32)])
@pytest.mark.parametrize("M,N", [(1, 16), (2, 33), (7, 100), (8, 260)])
def test_long_k(pkg, dev, M, N, K, g):
    import torch
    assert pkg.gemm_route(M, N, K, group_size=g) == "small_m"
    assert pkg.gemm_route(9, N, K, group_size=g) == "gemm"
    x, [(w, s, b)] = o.make_inputs(M, N, K, g, seed=M + N + K)
    x[M - 1, ::97] = np.inf      # a row of infinities and NaN stays in its row
    tx, args = to_dev(x, dev), [to_dev(a, dev) for a in (w, s, b)]
    y = pkg.matmul_q4_fast_f32(tx, *args, M, K, N, g).cpu().numpy()
    assert not np.isfinite(y[M - 1]).any()
    if M > 1:
        assert_parity(y[:-1], o.matmul_q4_f64(x[:-1], w, s, b, g), TOL_GEMM_F16, f"M={M} N={N} K={K}")
