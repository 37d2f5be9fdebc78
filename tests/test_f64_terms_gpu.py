"""The FP64 brute force term by term: as exact as IEEE square root and division, the same limits."""
import numpy as np
import pytest

import particular_amd as pa

pytestmark = pytest.mark.gpu


def errors(res, eps, m, reps):
    """Errors of the library's sums over m bodies and of a plain FP64 loop, in units of the terms' sum."""
    rng = np.random.default_rng(m)
    got, ieee = [], []
    for _ in range(reps):
        a, b = rng.normal(size=(512, 4)), rng.normal(size=(m, 4))
        b[:, 3] = np.abs(b[:, 3])
        d = b[None, :, :3] - a[:, None, :3]
        r2 = (d * d).sum(-1) + eps * eps
        plain = np.zeros((512, 3))
        for j in range(m):
            plain += d[:, j] * (b[j, 3] / (r2[:, j] * np.sqrt(r2[:, j])))[:, None]
        dl = b[None, :, :3].astype(np.longdouble) - a[:, None, :3]
        rl = (dl * dl).sum(-1) + np.longdouble(eps) ** 2
        term = dl * (b[None, :, 3] / (rl * np.sqrt(rl)))[..., None]
        scale = np.sqrt((term**2).sum(-1)).sum(1)
        mine = pa.BruteForce(res, pa.AccelerationSoftened.checked(eps)).compute(pa.Between(a, b))
        for out, x in ((got, mine), (ieee, plain)):
            out.append(np.sqrt(((x - term.sum(1)) ** 2).sum(1)) / scale)
    return [np.sqrt(np.mean(np.concatenate(e).astype(float) ** 2)) for e in (got, ieee)]


@pytest.mark.parametrize("eps", [0.0, 0.01, 0.3])
@pytest.mark.parametrize("m,reps", [(1, 64), (2, 64), (8, 64), (9, 32), (100, 8)])
def test_as_exact_as_ieee(res, eps, m, reps):
    """Root mean square error no larger than that of a square root, a product and a division per term;
    5 % for the sample (its own spread is below 1 %) and for the fused additions either side makes."""
    got, ieee = errors(res, eps, m, reps)
    assert got <= 1.05 * ieee


def one(res, x, mu, checked, eps=0.0):
    a, b = np.zeros((1, 4)), np.array([[x, 0.0, 0.0, mu]])
    with np.errstate(all="ignore"):
        return pa.BruteForce(res, pa.AccelerationSoftened(eps, checked)).compute(pa.Between(a, b))[0]


def test_vanishing_and_infinite_distances(res):
    """What d (mu / (r2 sqrt(r2))) gives: infinite where r2 or its cube vanishes, nothing where it
    overflows; checked, nothing where r2 vanishes."""
    for x in (1e-170, 1e-163, 1e-160, 1e-125):
        for mu in (1.0, -1.0):
            assert one(res, x, mu, False)[0] == mu * np.inf
            assert one(res, x, mu, True)[0] == (mu * np.inf if x > 1e-162 else 0.0)
    assert np.isnan(one(res, 0.0, 1.0, False)).all() and not one(res, 0.0, 1.0, True).any()
    for x in (1e150, 1e154, 1e160):
        for checked in (False, True):
            assert not one(res, x, 1.0, checked).any()


@pytest.mark.parametrize("eps", [0.0, 1e-20, 1e-3, 0.5])
@pytest.mark.parametrize("mu", [np.inf, 1e270])
def test_own_body_left_out(res, eps, mu):
    """Checked, a body adds nothing to itself or to one at its place, whatever its mu."""
    p = np.array([[0, 0, 0, mu], [1, 0, 0, 1.0], [0, 0, 0, 2.0]])
    got = pa.BruteForce(res, pa.AccelerationSoftened.checked(eps)).compute(p)
    want = 1 / (1 + eps * eps) ** 1.5
    np.testing.assert_allclose(got[[0, 2]], [[want, 0, 0]] * 2, rtol=1e-15)
    assert got[1, 0] == (-np.inf if np.isinf(mu) else pytest.approx(-mu * want, rel=1e-15))
