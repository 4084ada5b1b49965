"""The neighbour search of large segments by particle index against sorted order: the same lists and the same
trajectories, for a segment just over the limit, flat, folded and with crowded cells (blocks split at 32
sorted positions), beside smaller segments and on two streams."""
import numpy as np
import pytest

from velvet_amd import scenes as S
from velvet_amd.solver import ClothSolver

pytestmark = pytest.mark.gpu


def _scene(n, shape, seed):
    c = S.grid_cloth(n, 0.05, center=(0.3, 1.0, 0.2), jitter=2e-3, seed=seed, stream=20)
    x = c.x.astype(np.float64)
    if shape != "flat":
        z = x[:, 2] - x[:, 2].min()
        period = 4.0 if shape == "folded" else 0.5                     # few and many layers
        x[:, 2] = np.abs(z % (2 * period) - period)
        x[:, 1] += 0.04 * np.floor(z / period) % 0.2
    if shape == "crowded":
        x[:, 0] *= 0.5
    c.x = x.astype(np.float32)
    p = S.Params(num_substeps=2, num_iterations=1, tune_hash_grid=1)
    return S.Scene(S.finish_params(p, [c]), [c], [], 2)


def _run(scenes, **tuning):
    with ClothSolver(use_graph=False) as s:
        segs = [s.load_scene(sc) for sc in scenes]
        s.set_tuning(**tuning)
        for _ in range(2):
            s.Simulate()
        s.synchronize()
        out = []
        for k in segs:
            nb = s.read_hash(k)[-1]
            live = np.cumprod(nb != 0xFFFFFFFF, axis=0).astype(bool)
            out.append((s.positions(k), s.velocities(k), live, np.where(live, nb, 0)))
        return out


@pytest.mark.parametrize("shape,others,streams,grid", [("flat", (), 1, 0), ("folded", (20, 131), 1, 1),
                                                       ("crowded", (), 1, 1), ("folded", (200, 363), 2, 0)])
def test_by_index_equals_sorted(shape, others, streams, grid):
    print(f"[gpu] search order {shape} {others} streams={streams} grid={grid}", flush=True)
    scenes = [_scene(363, shape, 1)] + [_scene(n, "folded", 2 + k) for k, n in enumerate(others)]
    want = _run(scenes, neighbor_order=2, hash_grid=grid)
    got = _run(scenes, neighbor_order=0, streams=streams, hash_grid=grid)
    for a, b in zip(want, got):
        assert np.isfinite(a[0]).all() and a[2].any()
        for x, y in zip(a, b):
            assert np.array_equal(x, y)
