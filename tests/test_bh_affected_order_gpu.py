"""Affected particles in random order take no more walk steps than in the order of the whole key, also
where the root box is far wider than the dense part."""
import numpy as np
import pytest

import particular_amd as pa
from particular_amd import workloads

pytestmark = pytest.mark.gpu


def key_order(p):
    """Indices in the order of the 63-bit keys of the massive bodies' root box."""
    q = p[p[:, 3] != 0][:, :3].astype(np.float64)
    mn, mx = q.min(0), q.max(0)
    half = (mx - mn).max() / 2
    cell = (p[:, :3].astype(np.float64) - ((mn + mx) / 2 - half)) / (2 * half) * 2**21
    cell = np.clip(cell, 0, 2**21 - 1).astype(np.int64)
    key = np.zeros(len(p), np.int64)
    for b in range(21):
        for a in range(3):
            key |= ((cell[:, a] >> b) & 1) << (3 * b + a)
    return np.argsort(key, kind="stable")


@pytest.mark.parametrize("n", [16_384, 16_385, 100_003, 262_145, 600_000])
@pytest.mark.parametrize("cap,far", [(0.999, 0.0), (0.999, 1e4), (1 - 1e-12, 0.0)])
def test_steps(res, n, cap, far):
    """1 % covers the borders between wavefronts, which differ by the cells' ties."""
    pos, _ = workloads.plummer(n, seed=n, cap=cap)
    p = workloads.pack(pos, 1.0 / n)
    p[2 * n // 3 :, 3] = 0
    if far:
        p[0, :3] = far, 0, 0
    p = p[np.random.default_rng(n).permutation(n)]
    order = key_order(p)
    alg = pa.BarnesHut(res, 0.7, pa.Acceleration.checked())
    got = alg.compute(pa.Reordered.new(p))
    steps = pa.bh_stats(res)[0]
    ref = alg.compute(pa.Reordered.new(np.ascontiguousarray(p[order])))
    assert steps <= 1.01 * pa.bh_stats(res)[0]
    row = np.linalg.norm(got[order] - ref, axis=1)
    assert np.all(row <= 1e-5 * np.linalg.norm(ref, axis=1))
