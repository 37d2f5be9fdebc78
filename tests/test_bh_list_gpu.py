"""The batched Barnes-Hut walk against the stackless one (the form PNB_WALK_LANES names): the plain
walk's bits, the corrected walk to rounding, at the sizes where the batched walk changes form, and
with angles small enough that its node sequences outgrow their memory."""
import numpy as np
import pytest

import particular_amd as pa
from particular_amd import learned, metrics, workloads

pytestmark = pytest.mark.gpu


def both(res, monkeypatch, theta, storage, mlp=False):
    alg = pa.BarnesHut(res, theta, pa.Acceleration.checked(), mlp=mlp)
    got = alg.compute(storage)
    counted = pa.bh_stats(res)[1]
    monkeypatch.setenv("PNB_WALK_LANES", "64")
    ref = alg.compute(storage)
    assert counted == pa.bh_stats(res)[1]
    monkeypatch.delenv("PNB_WALK_LANES")
    return got, ref


@pytest.mark.parametrize("theta", [0.0, 0.12, 0.5, 1.3])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 17, 65, 1500, 6001])
def test_plain_bits(res, monkeypatch, n, theta):
    """Groups with idle lanes, single leaves, and (angles 0 and 0.12) sequences beyond their
    capacity, whose front is then walked node by node."""
    p = workloads.two_plummer_case(n, seed=n).particles
    got, ref = both(res, monkeypatch, theta, p)
    np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("n,m", [(17000, 17000), (40001, 25000), (3, 9000), (60000, 500)])
def test_two_sets_and_forms(res, monkeypatch, n, m):
    src = workloads.two_plummer_case(m, seed=m).particles
    a = workloads.two_plummer_case(n, seed=n + 1).particles
    a[: min(n, m) // 2] = src[: min(n, m) // 2]  # some at zero distance
    got, ref = both(res, monkeypatch, 0.6, pa.Between(a, src))
    np.testing.assert_array_equal(got, ref)


def test_coincident_and_deep(res, monkeypatch):
    """Runs of identical positions, chains of single-child nodes and a far outlier."""
    p = workloads.direct_sum_case(2000, seed=8).particles
    p[500:560, :3] = p[500, :3]
    p[600, :3] = p[601, :3] + np.float32(1e-6)
    p[0, :3] = 1e4
    got, ref = both(res, monkeypatch, 0.5, p)
    np.testing.assert_array_equal(got, ref)


def test_non_finite_affected(res, monkeypatch):
    """A particle with a non-finite position gets what the stackless walk gives it, and its
    neighbours are untouched."""
    src = workloads.direct_sum_case(3000, seed=9).particles
    a = src[:200].copy()
    a[7, 0] = np.nan
    a[90, 1] = np.inf
    alg = pa.BarnesHut(res, 0.5, pa.Acceleration.checked())
    got = alg.compute(pa.Between(a, src))
    monkeypatch.setenv("PNB_WALK_LANES", "64")
    ref = alg.compute(pa.Between(a, src))
    np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("params", ["quadrupole_params", "octupole_params"])
@pytest.mark.parametrize("n,theta", [(3, 0.5), (700, 0.1), (5000, 0.5), (30000, 0.6)])
def test_corrected_to_rounding(res, monkeypatch, params, n, theta):
    """The same terms in partial sums of other groups: the bar the stackless walk's own widths
    are held to."""
    p = workloads.two_plummer_case(n, seed=n).particles
    learned.init(res, 0)
    learned.set_params(res, getattr(learned, params)())
    got, ref = both(res, monkeypatch, theta, p, mlp=True)
    row = np.linalg.norm(got - ref, axis=1) / np.linalg.norm(ref, axis=1)
    assert metrics.rms_rel(got, ref) < 1e-6 and row.max() < 1e-5
