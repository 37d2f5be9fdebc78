"""Walks whose wavefronts start in the order of their expected work, around the sizes and angles where
that begins and ends: the plain walk's sums are those of the walk in tree order."""
import numpy as np
import pytest

import particular_amd as pa
from particular_amd import workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [229_375 - 64, 229_376, 262_145, 1_048_576, 1_048_577])
@pytest.mark.parametrize("theta", [0.7, 0.71])
def test_plain_bits(res, monkeypatch, n, theta):
    import torch

    p = workloads.two_plummer_case(n, seed=5).particles.copy()
    p[100:200, :3] = p[100, :3]  # a wavefront's box of no extent
    d = torch.from_numpy(p).cuda()
    alg = pa.BarnesHut(res, theta, pa.Acceleration.checked())
    got = alg.compute(d)
    monkeypatch.setenv("PNB_WALK_LANES", "32")  # not 64: no order
    ref = alg.compute(d)
    assert torch.equal(got[:, :3], ref[:, :3])


def test_non_finite_affected(res, monkeypatch):
    """Particles without a finite position get what the unordered walk gives them."""
    import torch

    p = workloads.two_plummer_case(300_000, seed=6).particles
    a = p.copy()
    a[5, 0], a[70_000, 1], a[200_000, 2] = np.nan, np.inf, -np.inf
    src, aff = torch.from_numpy(p).cuda(), torch.from_numpy(a).cuda()
    alg = pa.BarnesHut(res, 0.6, pa.Acceleration.checked())
    got = alg.compute(pa.Between(aff, src))[:, :3]
    monkeypatch.setenv("PNB_WALK_LANES", "32")
    ref = alg.compute(pa.Between(aff, src))[:, :3]
    assert torch.equal(got.isnan(), ref.isnan())
    assert torch.equal(got.nan_to_num(), ref.nan_to_num())
