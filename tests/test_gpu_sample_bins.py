"""The ends of the sampler's level-0 histogram: one bin per value of a
probability's top bits up to 1.0's, the last bin also taking NaN.  Against the
oracle (Ops.swift:2060-2098).

Every probability here is 0, 1, 1/2 or NaN, which both sides form exactly, so
the token must be the oracle's."""
import numpy as np
import pytest

from oracle import q4_oracle as o

pytestmark = pytest.mark.gpu


def _case(kind, n, dt):
    v = np.zeros(n, dt)
    if kind == "one":           # p = 1 and zeros
        v[:] = -1000
        v[n // 2] = 1000
    elif kind == "minus_inf":   # p = 1 and exact zeros from -inf
        v[:] = -np.inf
        v[n - 1] = 0
    elif kind == "two":         # p = 1/2 twice, zeros behind
        v[:] = -1000
        v[[1, n - 1]] = 4
    elif kind == "plus_inf":    # every p NaN
        v[n // 3] = np.inf
    elif kind == "all_minus_inf":
        v[:] = -np.inf
    elif kind == "one_nan":     # NaN in the middle of finite logits
        v[n // 2] = np.nan
    elif kind == "nan_signs":   # NaNs of both signs
        v[:] = np.nan
        v[::2] = -v[::2]
    return v


@pytest.mark.parametrize("kind", ["one", "minus_inf", "two", "plus_inf", "all_minus_inf",
                                  "one_nan", "nan_signs"])
@pytest.mark.parametrize("n", [2, 8192, 128256])   # within and beyond the LDS list
def test_level0_ends(pkg, dev, n, kind):
    import torch
    for dt in (np.float16, np.float32):
        lg = _case(kind, n, dt)
        x = torch.from_numpy(lg).to(dev)
        for top_p in (0.3, 0.9, 1.0):
            for u in (0.0, 0.25, 0.75, 0.9999):
                got = int(pkg.sample(x, 1.0, top_p, 1.0, None, u).item())
                with np.errstate(invalid="ignore"):
                    want = o.sample_ref(lg, 1.0, top_p, 1.0, [], u)
                assert got == want, (kind, n, dt.__name__, top_p, u, got, want)
