"""Host arrays through pinned memory and, above 1 MiB, through the runtime's copies: the same sums as
from device tensors, with one array on both sides, a prefix of it, and two arrays."""
import numpy as np
import pytest

import particular_amd as pa
from particular_amd import _lib

pytestmark = pytest.mark.gpu


def bodies(n, seed, dtype):
    p = np.random.default_rng(seed).normal(size=(n, 4)).astype(dtype)
    p[:, 3] = np.abs(p[:, 3]) + 0.1
    return p


@pytest.mark.parametrize("n,m", [(1, 1), (5, 3), (4096, 4096), (65536, 700), (65537, 700), (700, 65537)])
@pytest.mark.parametrize("one_array", [True, False])
def test_f32_host_sums_are_the_device_sums(res, n, m, one_array):
    import torch

    a = bodies(n, 1, np.float32)
    b = a[:m] if one_array and m <= n else bodies(m, 2, np.float32)
    inter = pa.AccelerationSoftened.checked(1e-2)
    for _ in range(2):
        host = pa.BruteForce(res, inter).compute(pa.Between(a, b))
        dev = pa.BruteForce(res, inter).compute(
            pa.Between(torch.from_numpy(a).cuda(), torch.from_numpy(b.copy()).cuda()))
        np.testing.assert_array_equal(host, dev.cpu().numpy()[:, :3])
        a = a[::-1].copy()  # other values in the same staging memory
        b = a[:m] if one_array and m <= n else b


@pytest.mark.parametrize("n,m", [(1, 1), (100, 100), (32768, 300), (32769, 300), (300, 32769)])
def test_f64_host_sums_are_the_device_sums(res, n, m):
    import torch

    a, b = bodies(n, 3, np.float64), bodies(m, 4, np.float64)
    host = pa.BruteForce(res, pa.AccelerationSoftened.checked(1e-2)).compute(pa.Between(a, b))
    da, db = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    out = torch.zeros((n, 4), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    res.use_torch_stream()
    res.check(_lib.lib().pnb_bf_accel_f64_dev(res.handle, da.data_ptr(), n, db.data_ptr(), m, 1e-2, 1,
                                              out.data_ptr()))
    torch.cuda.synchronize()
    np.testing.assert_array_equal(host, out.cpu().numpy()[:, :3])


@pytest.mark.parametrize("n", [2, 65536, 65537])
def test_pairs_host_sums_are_the_device_sums(res, n):
    import torch

    a = bodies(n, 5, np.float32)
    alg = pa.BruteForcePairs(res, pa.AccelerationSoftened.checked(1e-2))
    np.testing.assert_array_equal(alg.compute(a),
                                  alg.compute(torch.from_numpy(a).cuda()).cpu().numpy()[:, :3])


@pytest.mark.parametrize("n", [1, 3, 16383, 16384, 16385])
def test_step_states_read_back(res, n):
    """The leapfrog state read whole and array by array, around 1 MiB of results (16,384 bodies)."""
    p = bodies(n, 6, np.float64)
    mu = np.zeros(n, np.float32)
    mu[:5] = 1.0
    pos, vel = np.ascontiguousarray(p[:, :3]), np.ascontiguousarray(p[:, 1:])
    lib = _lib.lib()
    res.check(lib.pnb_leapfrog_init(res.handle, pos.ctypes.data, vel.ctypes.data, mu.ctypes.data, n, 1e-2, 1))
    x, v, a = np.empty((n, 3)), np.empty((n, 3)), np.empty((n, 4), np.float32)
    res.check(lib.pnb_leapfrog_read(res.handle, x.ctypes.data, v.ctypes.data, a.ctypes.data))
    np.testing.assert_array_equal(x, pos)
    np.testing.assert_array_equal(v, vel)
    f32 = np.concatenate([pos.astype(np.float32), mu[:, None]], 1)
    np.testing.assert_array_equal(
        a[:, :3], pa.BruteForce(res, pa.AccelerationSoftened.checked(1e-2)).compute(pa.Reordered.new(f32)))
    for k, whole in enumerate((x, v, a)):
        part = np.empty_like(whole)
        args = [None, None, None]
        args[k] = part.ctypes.data
        res.check(lib.pnb_leapfrog_read(res.handle, *args))
        np.testing.assert_array_equal(part, whole)


@pytest.mark.parametrize("n,m", [(5, 3), (4097, 4097), (65537, 1000), (1000, 65537)])
def test_barnes_hut_host_sums_are_the_device_sums(res, n, m):
    import torch

    a = bodies(n, 7, np.float32)
    b = a if n == m else bodies(m, 8, np.float32)
    alg = pa.BarnesHut(res, 0.6, pa.AccelerationSoftened.checked(1e-2))
    da = torch.from_numpy(a).cuda()
    dev = alg.compute(pa.Between(da, da if n == m else torch.from_numpy(b).cuda()))
    np.testing.assert_array_equal(alg.compute(pa.Between(a, b)), dev.cpu().numpy()[:, :3])
