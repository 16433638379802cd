"""nq_keep_mask at the sizes and value patterns where its selection can go wrong.

The reference result is exact: candidates sorted by value (descending), then by
position (ascending), the first k kept.  Sizes straddle the directly ranked
length (256 candidates), the 64-position runs of a lane, and the 16384-position
window; values cover one repeated value, few distinct values, a range one bin of
the histogram would hold, and the extremes of fp32.
"""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _values(kind, b, s, rng):
    if kind == "softmax":
        x = np.exp(rng.normal(-6.0, 4.0, (b, s)))
    elif kind == "constant":
        x = np.full((b, s), 0.125)
    elif kind == "few":
        x = rng.integers(0, 7, (b, s)) / 8.0
    elif kind == "narrow":  # neighbouring fp32 values: one first-pass bin holds many keys
        x = np.float32(1.0) + rng.integers(0, 5000, (b, s)) * np.float32(2.0 ** -23)
        x[:, ::997] = 1e30
    else:  # signs, infinities and the smallest values
        x = rng.normal(0.0, 1.0, (b, s)) * 10.0 ** rng.integers(-45, 38, (b, s))
        x[:, ::101] = np.inf
        x[:, ::211] = -np.inf
    return x.astype(np.float32)


def _expected(imp, rate, window, protected):
    from nexusquant_amd.ops import keep_plan
    b, s = imp.shape
    prefix, k = keep_plan(s, rate, window)
    keep = np.zeros((b, s), dtype=bool)
    keep[:, 0] = True
    if window > 0:
        keep[:, max(0, s - window):] = True
    for i in range(b):
        if k > 0:
            order = np.argsort(-imp[i, 1:prefix].astype(np.float64), kind="stable")
            keep[i, 1 + order[:k]] = True
    for p in protected:
        keep[:, p] = True
    return keep


@pytest.mark.parametrize("kind", ["softmax", "constant", "few", "narrow", "extreme"])
@pytest.mark.parametrize("s", [1, 2, 33, 65, 256, 289, 290, 1024, 4097, 16383, 16384, 16385, 32768, 50001, 131077])
def test_keep_mask_exact(s, kind):
    from nexusquant_amd.ops import keep_mask
    rng = np.random.default_rng(s)
    b = 2
    imp = _values(kind, b, s, rng)
    for rate, window, protected in ((0.6, 32, []), (0.05, 0, [0, s - 1, s // 2]), (0.999, 32, [s // 3])):
        keep, kept, n_kept = keep_mask(torch.from_numpy(imp).to(DEV), rate, window, protected or None)
        want = _expected(imp, rate, window, protected)
        got = keep.cpu().numpy().astype(bool)
        assert np.array_equal(got, want), (s, kind, rate)
        for i in range(b):
            yes, no = np.flatnonzero(want[i]), np.flatnonzero(~want[i])
            assert int(n_kept[i]) == yes.size
            assert np.array_equal(kept[i].cpu().numpy(), np.concatenate([yes, no[::-1]]))
