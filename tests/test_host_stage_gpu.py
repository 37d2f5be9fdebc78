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
