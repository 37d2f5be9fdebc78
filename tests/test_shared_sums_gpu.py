"""The workgroup-cooperative sums at the edges of their tiles and ranges."""
import ctypes

import numpy as np
import pytest

import particular_amd as pa
from particular_amd import _lib, metrics, workloads

pytestmark = pytest.mark.gpu


def bodies(n, seed):
    rng = np.random.default_rng(seed)
    p = rng.normal(size=(n, 4)).astype(np.float32)
    p[:, 3] = rng.uniform(0.5, 1.5, n)
    return p


@pytest.mark.parametrize("eps", [0.0, 1e-2])
@pytest.mark.parametrize("n,m", [(1, 65), (63, 1023), (64, 1024), (65, 1025), (129, 2048),
                                 (300, 4095), (70, 4097), (5, 40000), (2000, 16385), (33000, 257),
                                 (40000, 1001), (24577, 3000), (70001, 4100)])
def test_brute_force_edges(res, orc, n, m, eps):
    """Tiles of 64, 128 and 256 bodies, partial tiles, idle wavefronts and split ranges; FP32 pair
    terms are a few units in the last place from FP64, the bars those of the other brute-force
    tests."""
    a, b = bodies(n, n), bodies(m, m + 1)
    k = min(n, m, 7)
    b[:k, :3] = a[:k, :3]  # pairs at zero distance add nothing
    inter = pa.AccelerationSoftened.checked(eps) if eps else pa.Acceleration.checked()
    got = pa.BruteForce(res, inter).compute(pa.Between(a, b))
    idx = np.unique(np.concatenate([np.arange(min(n, 300)), np.arange(max(0, n - 300), n)]))
    ref = orc.direct_f64(a[idx], b, softening=eps)
    assert metrics.rms_rel(got[idx], ref) < 1e-5 and metrics.max_rel(got[idx], ref) < 1e-4


@pytest.mark.parametrize("n,eps", [(4500, 0.0), (7746, 1e-3), (7747, 1e-3), (24577, 0.0), (131075, 1e-3),
                                   (169999, 0.0), (239999, 1e-3)])
def test_pairs_below_the_pair_kernel(res, orc, n, eps):
    """Sets summed one-sided, each body's own term left out by index: with and without the mask."""
    import torch

    p = workloads.direct_sum_case(n, seed=n).particles
    inter = pa.AccelerationSoftened.checked(eps) if eps else pa.Acceleration.checked()
    dev = torch.from_numpy(p).cuda()
    got = pa.BruteForcePairs(res, inter).compute(dev).cpu().numpy()[:, :3]
    idx = np.random.default_rng(1).choice(n, 500, replace=False)
    ref = orc.direct_f64(p[idx], p, softening=eps)
    assert metrics.rms_rel(got[idx], ref) < 1e-5 and metrics.max_rel(got[idx], ref) < 1e-4


def test_pairs_own_term_only_is_left_out(res):
    """Unchecked and unsoftened: finite for distinct positions, non-finite exactly where two
    bodies coincide; a softening whose square vanishes leaves the own term out too."""
    p = workloads.direct_sum_case(9000, seed=3).particles
    assert np.all(np.isfinite(pa.BruteForcePairs(res, pa.Acceleration.unchecked()).compute(p)))
    tiny = pa.BruteForcePairs(res, pa.AccelerationSoftened.checked(1e-30)).compute(p)
    assert np.all(np.isfinite(tiny))
    p[8000] = p[17]
    bad = ~np.isfinite(pa.BruteForcePairs(res, pa.Acceleration.unchecked()).compute(p)).all(1)
    assert set(np.nonzero(bad)[0]) == {17, 8000}


def test_ensemble_by_workgroups_equals_single_systems(res):
    """Systems at the edges of tiles and groups, one large enough that the queue is taken by
    workgroups: the bits of the brute-force kernel on each system alone."""
    sizes = [1, 2, 63, 64, 65, 127, 255, 256, 257, 511, 513, 1025, 2047, 2049, 9001]
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    n = int(off[-1])
    pos, vel = workloads.plummer(n, 5)
    mu = np.random.default_rng(5).uniform(0.5, 1.5, n).astype(np.float32) / n
    L = _lib.lib()
    for eps in (0.0, 1e-3):
        res.reset_stream()
        res.check(L.pnb_batch_init(res.handle, pos.ctypes.data, vel.ctypes.data, mu.ctypes.data,
                                   off.ctypes.data, len(sizes), eps, 1))
        acc = np.zeros((n, 4), np.float32)
        res.check(L.pnb_batch_read(res.handle, None, None, acc.ctypes.data))
        res.set_bf_tuning(0, 1, 2, 1)
        try:
            for b, e in zip(off[:-1], off[1:]):
                p = workloads.pack(pos[b:e], mu[b:e])
                out = np.zeros((e - b, 4), np.float32)
                res.check(L.pnb_bf_accel_f32(res.handle, p.ctypes.data, e - b, p.ctypes.data, e - b,
                                             ctypes.c_float(eps), 1, out.ctypes.data))
                np.testing.assert_array_equal(acc[b:e], out)
        finally:
            res.clear_bf_tuning()
