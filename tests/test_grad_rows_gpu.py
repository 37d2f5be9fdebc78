"""The network's gradient over ragged training sets: wavefronts without rows, row counts around the
16-row tile, the 64-row mask and the 128-row chunk, and more tiles than the backward pass has
wavefronts. Against the FP64 oracle with the same bf16 rounding points."""
import numpy as np
import pytest

from oracle import mlp_oracle as M
from particular_amd import learned

pytestmark = pytest.mark.gpu


def ragged_set(seed, counts):
    rng = np.random.default_rng(seed)
    counts = np.asarray(counts)
    rows, waves = int(counts.sum()), len(counts)
    feats = np.zeros((rows, learned.FEAT), np.float32)
    feats[:, :M.IN] = rng.normal(size=(rows, M.IN))
    u = rng.normal(size=(rows, 3))
    geom = np.zeros((rows, learned.GEOM), np.float32)
    geom[:, :3] = 3.0 * u / np.linalg.norm(u, axis=1, keepdims=True)
    geom[:, 3] = rng.uniform(0.5, 2.0, rows)
    geom[:, 4] = geom[:, 3] * rng.uniform(0.5, 1.5, rows)
    lanes = np.zeros((waves, 64, 4), np.float32)
    lanes[..., :3] = rng.normal(size=(waves, 64, 3)) * 0.3
    lanes[..., 3] = 1e-4
    mask = rng.integers(0, 2**64, rows, dtype=np.uint64)
    mask[rng.random(rows) < 0.5] = np.uint64(2**64 - 1)
    return {"feats": feats, "geom": geom, "mask": mask,
            "row_wave": np.repeat(np.arange(waves), counts).astype(np.uint32),
            "wave_rows": np.concatenate([[0], np.cumsum(counts)]).astype(np.uint32),
            "lanes": lanes,
            "target": (rng.normal(size=(waves, 64, 4)) * 0.01).astype(np.float32),
            "wgt": rng.uniform(0.1, 1.0, (waves, 64)).astype(np.float32)}


@pytest.mark.parametrize("counts", [
    [1],
    [0, 1, 15, 16, 17, 0, 63, 64, 65, 127, 128, 129, 257, 0],
    [33, 700] * 45,  # 32,985 rows: 2,062 tiles for 2,048 wavefronts
])
def test_gradient_of_ragged_sets(res, counts):
    # The same rounding points on both sides: what is left is the bf16 values that FP32 sums round to
    # the other neighbour, 2^-8 of a few values each, and the FP32 sums themselves. 2e-2 of a
    # parameter array's norm and 1e-3 of the loss bound both.
    p = M.init_params(11)
    for k, n in (("b1", 64), ("b2", 64), ("b3", M.OUT)):
        p[k] = np.random.default_rng(n).normal(0, 0.1, n)
    p["W3"] = np.random.default_rng(12).normal(0, 0.1, (64, M.OUT))
    flat = learned.dict_to_params(p)
    learned.set_params(res, flat)
    p = learned.params_to_dict(flat.astype(np.float64))
    d = ragged_set(len(counts), counts)
    learned.clear(res)
    learned.load(res, d)
    loss, g = learned.grad(res)
    ref_loss, ref_g, _ = M.loss_and_grads(
        p, d["feats"][:, :M.IN].astype(np.float64), d["row_wave"].astype(np.int64), d["mask"],
        d["geom"].astype(np.float64), d["lanes"].astype(np.float64),
        d["target"][..., :3].astype(np.float64), d["wgt"].astype(np.float64), bf16=True)
    learned.clear(res)
    assert abs(loss / ref_loss - 1) < 1e-3
    gd = learned.params_to_dict(g)
    for k in ("W1", "b1", "W2", "b2", "W3", "b3"):
        assert np.linalg.norm(gd[k] - ref_g[k]) < 2e-2 * np.linalg.norm(ref_g[k]), k
