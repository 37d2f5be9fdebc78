"""The child table of the batched walk: written only where it pays, never asked of a capture."""
import numpy as np
import pytest
import torch

import particular_amd as pa
from particular_amd import learned, metrics, workloads
from tests.test_bh_graph_gpu import capture

pytestmark = pytest.mark.gpu


def cube(n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    p = torch.rand((n, 4), generator=g, device="cuda")
    p[:, 3] = 1.0 / n
    return p


@pytest.mark.parametrize("n,table", [(64, True), (65, False), (500, False), (1200, True)])
def test_few_probes_of_a_large_tree(monkeypatch, n, table):
    """2.8M nodes (90 MB of table): the plain walk's bits with or without it, and the memory it takes."""
    src = cube(2_000_000, 1)
    aff = src[::1000][:n].clone()
    out = torch.empty_like(aff)
    torch.cuda.synchronize()
    alg = pa.BarnesHut(None, 0.6, pa.Acceleration.checked())
    used = []
    for lanes in (None, "64"):
        if lanes:
            monkeypatch.setenv("PNB_WALK_LANES", lanes)  # a form of the stackless walk
        with pa.HipResources(0) as res:
            alg.resources = res
            res.use_torch_stream()
            free = torch.cuda.mem_get_info()[0]
            alg._between_dev(aff, src, out)
            torch.cuda.synchronize()
            used.append((free - torch.cuda.mem_get_info()[0], out[:, :3].clone()))
            nodes = len(pa.tree_export(res)[0])
    assert 2_000_000 < nodes < 2500 * 1200
    assert torch.equal(used[0][1], used[1][1])
    extra = used[0][0] - used[1][0]
    assert (extra > 24 * nodes) == table


def test_capture_of_the_trees_own_bodies():
    """Sized for many particles over a small tree, a capture of the small set on itself is taken, as
    eager calls of either are."""
    src, many = (torch.from_numpy(workloads.two_plummer_case(n, seed=n).particles).cuda() for n in (3000, 80_000))
    alg = pa.BarnesHut(None, 0.5, pa.Acceleration.checked())
    with pa.HipResources(0) as res:
        alg.resources = res
        own, two = alg.compute(src), alg.compute(pa.Between(many, src))
        res.set_bh_capturable(True)
        alg.compute(pa.Between(many, src))  # sizes
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with capture(graph):
            got = alg.compute(pa.Between(src, src))
        for _ in range(2):
            again = alg.compute(pa.Between(many, src))
            torch.cuda.synchronize()
            assert torch.equal(again, two)
            got.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(got, own)
        res.bh_check()


@pytest.mark.parametrize("params", ["quadrupole_params", "octupole_params"])
@pytest.mark.parametrize("n,theta,batched", [(40_000, 1.3, True), (40_001, 1.3, False), (78_000, 0.6, True),
                                             (79_000, 0.6, False), (150_000, 0.3, True), (150_001, 0.3, False)])
def test_corrected_borders(monkeypatch, params, n, theta, batched):
    """Both sides of the border between the walks, which falls with the angle: the same accepted nodes,
    sums to rounding (the bar the stackless walk's own widths are held to), and the walk it should be
    (the batched one adds the same terms in other groups; the stackless one's bits repeat)."""
    p = workloads.two_plummer_case(n, seed=n).particles
    with pa.HipResources(0) as res:
        learned.init(res, 0)
        learned.set_params(res, getattr(learned, params)())
        alg = pa.BarnesHut(res, theta, pa.Acceleration.checked(), mlp=True)
        got, counted = alg.compute(p), pa.bh_stats(res)[1]
        steps = pa.bh_stats(res)[0]
        lanes = 64
        while lanes > 1 and -(-n // lanes) < 2048:
            lanes //= 2
        monkeypatch.setenv("PNB_WALK_LANES", str(lanes))
        ref = alg.compute(p)
        assert counted == pa.bh_stats(res)[1]
        assert (steps == pa.bh_stats(res)[0]) != batched
    if not batched:
        np.testing.assert_array_equal(got, ref)
    row = np.linalg.norm(got - ref, axis=1) / np.linalg.norm(ref, axis=1)
    assert metrics.rms_rel(got, ref) < 1e-6 and row.max() < 1e-5


def test_capture_at_another_angle():
    """Sized at an angle without a child table, a capture at one that would want it is taken."""
    d = torch.from_numpy(workloads.two_plummer_case(70_000, seed=2).particles).cuda()
    with pa.HipResources(0) as res:
        learned.init(res, 0)
        learned.set_params(res, learned.quadrupole_params())
        wide, narrow = (pa.BarnesHut(res, th, pa.Acceleration.checked(), mlp=True) for th in (0.9, 0.4))
        res.set_bh_capturable(True)
        wide.compute(pa.Between(d, d))  # sizes
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with capture(graph):
            got = narrow.compute(pa.Between(d, d))
        for _ in range(2):
            eager = narrow.compute(pa.Between(d, d))
            torch.cuda.synchronize()
            got.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(got, eager) and bool(torch.isfinite(got).all())
        res.bh_check()
