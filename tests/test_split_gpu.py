"""The split of a device tensor's massive particles at the sizes where its launches change: a
workgroup's turn of 1,024, one workgroup, and more than 1,024 workgroups' turns. The sums over the
split are those over the massive particles taken out on the host, in their order."""
import numpy as np
import pytest

import particular_amd as pa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 1023, 1024, 1025, 5000, 1 << 20, (1 << 20) + 1, 2_500_001])
@pytest.mark.parametrize("massive", ["few", "first", "last", "none"])
def test_split_keeps_the_massive_in_order(res, n, massive):
    import torch

    rng = np.random.default_rng(n)
    p = rng.normal(size=(n, 4)).astype(np.float32)
    p[:, 3] = 0.0
    some = {"few": rng.choice(n, min(n, 300), replace=False), "first": np.arange(min(n, 70)),
            "last": np.arange(max(0, n - 70), n), "none": np.arange(0)}[massive]
    p[some, 3] = rng.uniform(0.5, 1.5, len(some))
    d = torch.from_numpy(p).cuda()
    alg = pa.BruteForce(res, pa.AccelerationSoftened.checked(1e-2))
    got = alg.compute(pa.Reordered.new(d))
    if massive == "none":
        assert not got[:, :3].any()
        return
    ref = alg.compute(pa.Between(d, torch.from_numpy(p[p[:, 3] != 0.0].copy()).cuda()))
    assert torch.equal(got[:, :3], ref[:, :3])


def test_split_of_all_massive(res):
    import torch

    p = np.random.default_rng(1).uniform(0.5, 1.5, size=(2049, 4)).astype(np.float32)
    p[7, 3] = np.nan  # not zero: massive
    d = torch.from_numpy(p).cuda()
    alg = pa.BruteForce(res, pa.AccelerationSoftened.checked(1e-2))
    a, b = alg.compute(pa.Reordered.new(d))[:, :3], alg.compute(pa.Between(d, d))[:, :3]
    assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num())
