"""The GEMM's fast kernel at group sizes 32 and 128 (scale / bias dwords copied
direct to LDS) and both its weight-tile widths against its generic kernel,
which stages them through registers and which a scale array at an odd 2-byte
address selects.  Both dequantize alike; K splits and the halves of the
128-row weight tiles may add the fp32 sums in another order.  An output is
K / 16 MFMA steps, each rounding a partial sum of at most about the largest
output once, on either side: the difference is bounded by
2 (K / 16) 2^-24 max|y| (fp16 outputs: one more half ulp on either side).  The
generic kernel is held to the oracle in test_gpu_gemm.py; one case here is too.

K covers one and several super-stages (128 k), odd counts of them, and at
group 128 splits that begin on the second group of a scale dword; M and N
cover partial tiles, split, single-round and persistent launches.  bf16
activations run the GEMM at every shape; fp16 ones take the wide-M route where
its grid is one round, so TILES names shapes where they run the GEMM, at each of
its tiles."""
import numpy as np
import pytest

from helpers import TOL_GEMM_F16, assert_parity, gpu_inputs, host, plan
from oracle import q4_oracle as o

pytestmark = pytest.mark.gpu


def _odd(t):
    """The same values at an address 2 bytes past a multiple of 4."""
    import torch
    buf = torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)
    v = buf[1:1 + t.numel()].view(t.shape)
    v.copy_(t)
    assert v.data_ptr() % 4 == 2
    return v


def _close(a, b, K, half=False):
    a, b = a.double(), b.double()
    tol = 2 * (K / 16) * 2.0**-24 * b.abs().max() + (2.0**-10 * b.abs() if half else 0.0)
    return bool(((a - b).abs() <= tol).all())


# (300, 500, 1280) splits K; (1000, 16384, 512) runs persistent blocks
SHAPES = [(257, 256, 256), (300, 500, 1280), (300, 777, 3328), (513, 3072, 3072), (700, 1000, 768),
          (1000, 16384, 512),
          # 128-row weight tiles: one round, partial tiles; three K splits (bf16)
          (700, 5000, 1280), (1537, 2040, 2304), (300, 2048, 2560)]


# (M, N, K, activation and weight rows of a tile, K splits, persistent)
TILES = [(257, 6000, 256, 128, 128, 1, False), (300, 3000, 4352, 128, 128, 3, False),
         (513, 7000, 256, 128, 256, 1, False), (130, 9000, 2304, 128, 256, 3, False),
         (700, 16500, 256, 128, 256, 1, True), (1537, 5000, 256, 192, 256, 1, False),
         (130, 9000, 4352, 192, 256, 7, False), (900, 16500, 512, 192, 256, 1, True)]
PAIR_TILES = [(257, 3000, 256, 128, 128, 1, False), (300, 1500, 4352, 128, 128, 3, False),
              (257, 6000, 256, 128, 256, 1, False), (257, 1500, 4352, 128, 256, 7, False),
              (400, 12300, 256, 128, 256, 1, True), (513, 7000, 256, 192, 256, 1, False),
              (130, 6000, 4352, 192, 256, 5, False), (900, 9000, 256, 192, 256, 1, True)]


def _runs_tile(pkg, M, N, K, g, pair, rows, wrows, splits, persistent):
    tiles = -(-M // rows) * -(-N // (wrows // 2 if pair else wrows))
    return (plan(pkg, M, N, K, g, pair) == ("gemm", splits, rows, wrows) and
            persistent == (splits == 1 and tiles > 256))


@pytest.mark.parametrize("g", [32, 64, 128])
@pytest.mark.parametrize("M,N,K,rows,wrows,splits,persistent", TILES)
def test_f16_tiles_equal_generic(pkg, dev, M, N, K, g, rows, wrows, splits, persistent):
    import torch
    assert _runs_tile(pkg, M, N, K, g, False, rows, wrows, splits, persistent)
    x, [(w, s, b)] = gpu_inputs(M, N, K, g, seed=M + N + K, dev=dev)
    fast = pkg.matmul_q4_fast_f32(x, w, s, b, M, K, N, g)
    gen = pkg.matmul_q4_fast_f32(x, w, _odd(s), _odd(b), M, K, N, g)
    torch.cuda.synchronize()
    assert _close(fast, gen, K)
    rows = np.array([0, 127, 128, M - 1])
    ref = o.matmul_q4_f64(host(x)[rows].astype(np.float64), host(w), host(s), host(b), g)
    assert_parity(fast.cpu().numpy()[rows], ref, TOL_GEMM_F16, f"g={g}")


@pytest.mark.parametrize("g", [32, 64, 128])
@pytest.mark.parametrize("M,N,K,rows,wrows,splits,persistent", PAIR_TILES)
def test_pair_tiles_equal_generic(pkg, dev, M, N, K, g, rows, wrows, splits, persistent):
    import torch
    assert _runs_tile(pkg, M, N, K, g, True, rows, wrows, splits, persistent)
    x, sets = gpu_inputs(M, N, K, g, seed=M + K, dev=dev, n_weights=2)
    fast = pkg.matmul_q4_silu_mul(x, *(pkg.Q4Weight(*t, K, g) for t in sets), M, K, N)
    gen = pkg.matmul_q4_silu_mul(x, *(pkg.Q4Weight(w, _odd(s), _odd(b), K, g) for w, s, b in sets),
                                 M, K, N)
    torch.cuda.synchronize()
    assert _close(fast, gen, K, half=True)


@pytest.mark.parametrize("g", [32, 64, 128])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_fast_equals_generic(pkg, dev, M, N, K, g):
    import torch
    for dt in ("f16", "bf16"):
        x, [(w, s, b)] = gpu_inputs(M, N, K, g, seed=M + N + K, dev=dev, x_dtype=dt)
        fast = pkg.matmul_q4_ex(x, pkg.Q4Weight(w, s, b, K, g), M, N)
        gen = pkg.matmul_q4_ex(x, pkg.Q4Weight(w, _odd(s), _odd(b), K, g), M, N)
        torch.cuda.synchronize()
        assert _close(fast, gen, K), f"{dt} M={M} N={N} K={K} g={g}"


@pytest.mark.parametrize("g", [32, 128])
@pytest.mark.parametrize("M,N,K", [(300, 200, 512), (700, 8192, 768), (500, 384, 3072), (200, 8000, 1280)])
def test_fast_equals_generic_pair(pkg, dev, M, N, K, g):
    import torch
    x, sets = gpu_inputs(M, N, K, g, seed=M + K, dev=dev, n_weights=2)
    fast = pkg.matmul_q4_silu_mul(x, *(pkg.Q4Weight(*t, K, g) for t in sets), M, K, N)
    gen = pkg.matmul_q4_silu_mul(x, *(pkg.Q4Weight(w, _odd(s), _odd(b), K, g) for w, s, b in sets),
                                 M, K, N)
    torch.cuda.synchronize()
    assert _close(fast, gen, K, half=True)


@pytest.mark.parametrize("g", [32, 128])
def test_fast_oracle(pkg, dev, g):
    import torch
    M, N, K = 400, 600, 1280
    x, [(w, s, b)] = gpu_inputs(M, N, K, g, seed=g, dev=dev)
    y = pkg.matmul_q4_fast_f32(x, w, s, b, M, K, N, g)
    torch.cuda.synchronize()
    rows = np.array([0, 127, 128, M - 1])
    ref = o.matmul_q4_f64(host(x)[rows].astype(np.float64), host(w), host(s), host(b), g)
    assert_parity(y.cpu().numpy()[rows], ref, TOL_GEMM_F16, f"g={g}")
