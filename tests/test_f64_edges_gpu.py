"""The FP64 brute force at the edges of its workgroups and ranges, and at extreme distances."""
import numpy as np
import pytest

import particular_amd as pa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(1, 1), (63, 3), (64, 255), (65, 513), (1000, 4097), (20000, 700),
                                 (3, 20000)])
@pytest.mark.parametrize("eps", [0.0, 1e-25, 0.03])
def test_f64_edges(res, n, m, eps):
    """Against numpy in extended precision; the bar covers a few units in the last place of every
    term and the summation of up to 20,000 of them."""
    rng = np.random.default_rng(n + m)
    a, b = rng.normal(size=(n, 4)), rng.normal(size=(m, 4))
    k = min(n, m, 5)
    b[:k, :3] = a[:k, :3]
    got = pa.BruteForce(res, pa.AccelerationSoftened.checked(eps)).compute(pa.Between(a, b))
    idx = np.unique(np.concatenate([np.arange(min(n, 40)), np.arange(max(0, n - 40), n)]))
    d = b[None, :, :3].astype(np.longdouble) - a[idx, None, :3]
    r2 = (d * d).sum(-1)
    s = np.where(r2 > 0, b[None, :, 3] / np.where(r2 > 0, r2 + np.longdouble(eps) ** 2, 1) ** 1.5, 0)
    term = d * s[..., None]
    err = np.abs(got[idx] - term.sum(1)).max(1)
    assert np.all(err <= 2e-15 * np.abs(term).sum((1, 2)) + 1e-300)


def test_f64_extremes(res):
    """Distances whose squares vanish or overflow, as IEEE square root and division give them."""
    a = np.array([[0.0, 0.0, 0.0, 0.0]])
    for x, want in ((1e-160, np.inf), (1e160, 0.0), (1e100, 1e-200)):
        b = np.array([[x, 0.0, 0.0, 1.0]])
        got = pa.BruteForce(res, pa.Acceleration.unchecked()).compute(pa.Between(a, b))
        if np.isfinite(want) and want > 0:
            np.testing.assert_allclose(got[0, 0], want, rtol=1e-14)
        else:
            assert not np.isnan(got[0, 1]) or want == np.inf
            assert got[0, 0] == want or (want == np.inf and not np.isfinite(got[0, 0]))
