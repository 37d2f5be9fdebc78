"""Scratch of one entry point stays valid when another one's grows: kept and captured graphs."""
import numpy as np
import pytest
import torch

import particular_amd as pa
from particular_amd import _lib, workloads
from tests.test_bh_graph_gpu import capture
from tests.test_step_gpu import init, read, run

pytestmark = pytest.mark.gpu


def grow_others(res):
    """Calls that size the split sums of the FP64, the pair and the f32 brute force."""
    rng = np.random.default_rng(3)
    p = torch.from_numpy(rng.normal(size=(130000, 4)).astype(np.float32)).cuda()
    pa.BruteForce(res, pa.Acceleration.checked()).compute(rng.normal(size=(10007, 4)))
    pa.BruteForcePairs(res, pa.AccelerationSoftened.checked(1e-2)).compute(p)
    pa.BruteForce(res, pa.AccelerationSoftened.checked(1e-2)).compute(pa.Between(p, p[:70000]))
    res.reset_stream()


def test_leapfrog_graph_after_other_calls():
    """The kept graph of a step loop replayed after other calls on the handle grew their scratch, and
    after a tuning entry that splits the loop's own sums further: the eager loop's bits."""
    s = workloads.massive_massless_case(n_massive=16384, n_total=65536)
    with pa.HipResources(0) as kept, pa.HipResources(0) as eager:
        init(kept, s)
        init(eager, s)
        run(kept, 2, 1e-3, True)
        run(eager, 2, 1e-3, False)
        grow_others(kept)
        run(kept, 2, 1e-3, True)
        run(eager, 2, 1e-3, False)
        for a, b in zip(read(kept, s.n), read(eager, s.n)):
            np.testing.assert_array_equal(a, b)
        for r in (kept, eager):
            r.check(_lib.lib().pnb_bf_set_tuning(r.handle, 1, 1, 1, 32))
        run(kept, 3, 1e-3, False)
        run(kept, 2, 1e-3, True)
        run(eager, 5, 1e-3, False)
        for a, b in zip(read(kept, s.n), read(eager, s.n)):
            np.testing.assert_array_equal(a, b)


def test_f64_graph_holds_no_scratch(res):
    """An FP64 sum captured by the caller and replayed after eager sums of another size: the same bits
    each time, and the eager result but for the order of its 3,000 positive terms' roundings."""
    rng = np.random.default_rng(1)
    a = torch.from_numpy(np.abs(rng.normal(size=(3000, 4)))).cuda()
    big = torch.from_numpy(rng.normal(size=(20000, 4))).cuda()
    out, out_big = torch.zeros_like(a), torch.zeros_like(big)

    def call(x, o):
        res.use_torch_stream()
        res.check(_lib.lib().pnb_bf_accel_f64_dev(res.handle, x.data_ptr(), x.shape[0], x.data_ptr(),
                                                  x.shape[0], 1e-3, 1, o.data_ptr()))

    call(a, out)
    torch.cuda.synchronize()
    want = out.clone()
    graph = torch.cuda.CUDAGraph()
    with capture(graph):
        call(a, out)
    first = None
    for _ in range(3):
        call(big, out_big)
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        first = out.clone() if first is None else first
        assert torch.equal(out, first)
    term = torch.linalg.vector_norm(want[:, :3], dim=1)
    assert float(((first - want).abs().max(1).values / term).median()) <= 1e-12


def test_host_staging_after_a_failed_call():
    """Host arrays staged right after a call that failed behind its own staging, on another stream: the
    sums of the new arrays."""
    rng = np.random.default_rng(4)
    p, q = (np.abs(rng.normal(size=(60_000, 4))).astype(np.float32) for _ in range(2))
    with pa.HipResources(0) as fresh, pa.HipResources(0) as res:
        alg, corrected = (pa.BarnesHut(res, 0.7, pa.Acceleration.checked(), mlp=m) for m in (False, True))
        want = pa.BarnesHut(fresh, 0.7, pa.Acceleration.checked()).compute(q)
        streams = [torch.cuda.Stream() for _ in range(2)]
        for k in range(20):
            res.set_stream(streams[k % 2].cuda_stream)
            with pytest.raises(pa.PnbError):  # no network
                corrected.compute(p)
            res.set_stream(streams[1 - k % 2].cuda_stream)
            np.testing.assert_array_equal(alg.compute(q), want)
        res.reset_stream()
