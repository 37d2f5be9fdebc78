"""The octree against the oracle at the sizes where the build changes its launches: one workgroup's
turn of 1,024 bodies, the single launches of the counts (2,048), of their scan and of the root box
(16,384), with runs of equal positions across the seams."""
import pytest

import particular_amd as pa
from particular_amd import workloads
from .treecheck import assert_same_tree, bh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1023, 1024, 1025, 2047, 2048, 2049, 4097, 16383, 16384, 16385])
def test_tree_at_the_builds_sizes(res, orc, m):
    p = workloads.two_plummer_case(m, seed=m).particles.copy()
    p[m // 3: m // 3 + 70, :3] = p[m // 3, :3]  # a run longer than a wavefront
    p[-1, :3] = p[0, :3]
    for _ in range(2):
        bh(res, pa.Between(p[:1], p), 0.5)
        assert_same_tree(res, orc, p)
