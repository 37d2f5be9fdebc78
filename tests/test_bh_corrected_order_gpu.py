"""Corrected walks whose wavefronts start in the order of their expected work, around the counts where
that begins and ends: the bits of the walk in tree order, which a capturable build keeps."""
import pytest

import particular_amd as pa
from particular_amd import learned, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("params", ["quadrupole_params", "octupole_params"])
@pytest.mark.parametrize("n", [163_840 - 64, 163_840 - 63, 300_001, 2_080_768, 2_080_769])
def test_corrected_bits(params, n):
    import torch

    p = workloads.two_plummer_case(n, seed=7).particles.copy()
    p[100:200, :3] = p[100, :3]  # a wavefront's box of no extent
    d = torch.from_numpy(p).cuda()
    with pa.HipResources(0) as res:
        learned.init(res, 0)
        learned.set_params(res, getattr(learned, params)())
        alg = pa.BarnesHut(res, 0.8, pa.Acceleration.checked(), mlp=True)
        got = alg.compute(d)
        steps = pa.bh_stats(res)[0]
        res.set_bh_capturable(True)
        alg.compute(d)  # sizes
        ref = alg.compute(d)
        res.bh_check()
        assert steps == pa.bh_stats(res)[0]
        assert torch.equal(got, ref)


def test_plain_two_sets():
    """The order also where the affected particles are not the tree's, with a ragged last wavefront."""
    import torch

    src = torch.from_numpy(workloads.two_plummer_case(100_000, seed=8).particles).cuda()
    aff = torch.from_numpy(workloads.two_plummer_case(300_017, seed=9).particles).cuda()
    with pa.HipResources(0) as res:
        alg = pa.BarnesHut(res, 0.6, pa.Acceleration.checked())
        got = alg.compute(pa.Between(aff, src))
        res.set_bh_capturable(True)
        alg.compute(pa.Between(aff, src))
        assert torch.equal(got, alg.compute(pa.Between(aff, src)))
