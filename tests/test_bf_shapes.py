"""How the brute-force sums are divided: every count the entry points take fits one dispatch."""
import os
import subprocess

import numpy as np
import pytest

import particular_amd as pa
from particular_amd import _lib, metrics

CSRC = os.path.join(os.path.dirname(pa.__file__), "csrc")

CHECK = r"""
#include "bf_shape.hpp"
#include <algorithm>
#include <cstdio>
#include <vector>
using namespace pnb;
int main() {
    const size_t limit = 0xffffffffu, top = 0x7fffffffu;
    std::vector<size_t> ns, ms;
    for (int k = 0; k <= 31; ++k)
        for (long d = -1; d <= 1; ++d) {
            const size_t v = (size_t(1) << k) + d;
            if (v >= 1 && v <= top) { ns.push_back(v); ms.push_back(v); }
        }
    for (size_t m : {100, 129, 200, 257, 300, 500, 700, 1000, 1500, 2047}) ms.push_back(m);
    for (size_t cus : {1, 32, 256, 304})
        for (size_t n : ns)
            for (size_t m : ms) {
                const BfPlan p = plan_for(default_shape(cus, n, m), m);
                const size_t x = bf_grid_x(p.shape, n), block = bf_block(p.shape);
                const size_t covered = x * (p.shape.variant == BF_COOP ? 64 : block * p.shape.per_lane);
                const bool all = covered >= n && size_t(p.splits) * p.chunk >= m &&
                                 size_t(p.splits - 1) * p.chunk < m;
                // few affecting bodies leave wavefronts of the cooperative kernel without a tile: only
                // where the affected ones cannot fill the chip by themselves
                if (cus == 256 && m <= 448 && n >= 262144 && p.shape.variant == BF_COOP) return 2;
                const Bf64Plan q = plan64(cus, n, m);
                const size_t x64 = ceil_div(std::min(n, BF64_SLICE), 64);
                const bool all64 = q.splits * q.chunk >= m && (q.splits == 1 || n <= BF64_SLICE);
                if (!all || !all64 || x * block > limit || x64 * 64 * BF64_WAVES > limit) {
                    std::printf("%zu CUs, %zu affected, %zu affecting: %zu x %zu\n", cus, n, m, x, block);
                    return 1;
                }
            }
    return 0;
}
"""


def test_launches_fit_a_dispatch(tmp_path):
    """Work-items along x stay below 2^32 and the workgroups cover both sides, at every power of two
    and beside it up to 2^31 - 1, the most the entry points take."""
    src, exe = tmp_path / "shapes.cpp", tmp_path / "shapes"
    src.write_text(CHECK)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("eps", [0.0, 1e-2])
@pytest.mark.parametrize("n,m", [(200_000, 257), (200_001, 257), (262_144, 448), (262_145, 449), (399_999, 200),
                                 (400_000, 200), (400_001, 263), (799_999, 449), (800_000, 449),
                                 (1_000_003, 511), (1_000_003, 513), (1_000_003, 2047), (300_001, 4103)])
def test_few_affecting(res, orc, n, m, eps):
    """Both sides of the borders between the kernels for few affecting bodies, and tiles that end in
    0 to 7 of them: the bars of the other brute-force tests."""
    rng = np.random.default_rng(m)
    a, b = (rng.normal(size=(k, 4)).astype(np.float32) for k in (n, m))
    b[:, 3] = rng.uniform(0.5, 1.5, m)
    b[:7, :3] = a[:7, :3]  # pairs at zero distance add nothing
    inter = pa.AccelerationSoftened.checked(eps) if eps else pa.Acceleration.checked()
    got = pa.BruteForce(res, inter).compute(pa.Between(a, b))
    idx = np.concatenate([np.arange(300), np.arange(n - 300, n)])
    ref = orc.direct_f64(a[idx], b, softening=eps)
    assert metrics.rms_rel(got[idx], ref) < 1e-5 and metrics.max_rel(got[idx], ref) < 1e-4


@pytest.mark.gpu
@pytest.mark.parametrize("first", [1, 2, 3, 5])
@pytest.mark.parametrize("n,m", [(300, 1100), (5000, 4099), (300_000, 2500)])
def test_slices(res, first, n, m):
    """Arrays that begin at any body of a larger one: the bits of a copy."""
    import torch

    g = torch.Generator(device="cuda").manual_seed(n)
    a, b = (torch.randn((k + 8, 4), generator=g, device="cuda")[first : first + k] for k in (n, m))
    alg = pa.BruteForce(res, pa.AccelerationSoftened.checked(1e-2))
    assert torch.equal(alg.compute(pa.Between(a, b)), alg.compute(pa.Between(a.clone(), b.clone())))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,n,m", [("f32", (1 << 28) + 67, 300), ("f64", (1 << 29) + 67, 3)])
def test_most_affected(res, dtype, n, m):
    """Counts whose cooperative (f32) and single (FP64) launch would hold 2^32 work-items or more.
    Rows at both ends and across the FP64 launches' border against numpy: the FP32 bar is 300 terms of
    a few units in the last place each, the FP64 one a few units in the last place."""
    import torch

    t = torch.float32 if dtype == "f32" else torch.float64
    if torch.cuda.mem_get_info()[0] < 3 * n * 4 * t.itemsize:
        pytest.skip("not enough free device memory")
    g = torch.Generator(device="cuda").manual_seed(2)
    a = torch.rand((n, 4), generator=g, device="cuda", dtype=t)
    b = torch.rand((m, 4), generator=g, device="cuda", dtype=t) + 0.5
    out = torch.full((n, 4), 7.0, device="cuda", dtype=t)
    fn = getattr(_lib.lib(), f"pnb_bf_accel_{dtype}_dev")
    res.use_torch_stream()
    res.check(fn(res.handle, a.data_ptr(), n, b.data_ptr(), m, 0.25, 1, out.data_ptr()))
    torch.cuda.synchronize()
    rows = np.unique(np.concatenate([np.arange(70), n - 1 - np.arange(70),
                                     (1 << 28) + np.arange(-70, 70 if n > (1 << 28) + 70 else 60)]))
    idx = torch.from_numpy(rows).cuda()
    x, y, got = (v.cpu().double().numpy() for v in (a[idx], b, out[idx]))
    d = y[None, :, :3] - x[:, None, :3]
    term = d * (y[None, :, 3] * ((d * d).sum(-1) + 0.0625) ** -1.5)[..., None]
    bar = (2e-6 if dtype == "f32" else 4e-15) * np.abs(term).sum(1)
    assert np.all(np.abs(got[:, :3] - term.sum(1)) <= bar)
    assert np.all(got[:, 3] == 0)
    assert float(out[:, 3].abs().max()) == 0  # no row left as it was
