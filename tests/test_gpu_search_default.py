"""The default search order (neighbor_order 2) of a grid cloth of more than 2^19 particles on a tuned hash grid:
by particle index while its cells are sparsely filled, in sorted order where they are crowded. The same
lists and trajectories as in sorted order either way, and at rest faster than it (the search by index takes
two thirds of the time; required: no more than 0.85)."""
import json

import numpy as np
import pytest

from velvet_amd import scenes as S
from velvet_amd.solver import ClothSolver

pytestmark = pytest.mark.gpu


def _scene(n, squeeze=1.0):
    c = S.grid_cloth(n, 0.01, center=(0.3, 1.0, 0.2), jitter=1e-4, seed=n, stream=20)
    c.x[:, 0] *= np.float32(squeeze)
    p = S.Params(num_substeps=2, num_iterations=1, tune_hash_grid=1)
    return S.Scene(S.finish_params(p, [c]), [c], [], 2)


def _run(scenes, streams, **tuning):
    with ClothSolver(use_graph=False) as s:
        segs = [s.load_scene(sc) for sc in scenes]
        s.set_tuning(streams=streams, **tuning)
        for _ in range(2):
            s.Simulate()
        s.synchronize()
        out = []
        for k in segs:
            nb = s.read_hash(k)[-1]
            live = np.cumprod(nb != 0xFFFFFFFF, axis=0).astype(bool)
            out.append((s.positions(k), s.velocities(k), live, np.where(live, nb, 0)))
        s.set_timing(True)
        for _ in range(3):
            s.Simulate()
        return out, json.loads(s.timing())["Solver_HashCache"]["ms"]


@pytest.mark.parametrize("n,squeeze,others,streams,grid", [(724, 1.0, (), 1, 1), (725, 1.0, (), 1, 2), (725, 0.5, (40,), 1, 1),
                                                           (730, 0.7, (363, 50), 2, 3), (725, 0.01, (), 1, 1)])
def test_default_equals_sorted(n, squeeze, others, streams, grid):
    print(f"[gpu] default search n={n} squeezed to {squeeze} grid={grid}", flush=True)
    scenes = [_scene(n, squeeze)] + [_scene(k) for k in others]
    want, _ = _run(scenes, 1, neighbor_order=1, hash_grid=grid)
    got, _ = _run(scenes, streams, hash_grid=grid)
    for a, b in zip(want, got):
        assert np.isfinite(a[0]).all() and a[2].any()
        for x, y in zip(a, b):
            assert np.array_equal(x, y)


def test_time_at_rest():
    scenes = [_scene(1024)]
    t = [min(_run(scenes, 1, neighbor_order=o, hash_grid=2)[1] for _ in range(2)) for o in (1, 2)]
    print(f"[gpu] searches of 1,048,576 particles: {t[0]:.3f} ms sorted, {t[1]:.3f} ms by default", flush=True)
    assert t[1] < 0.85 * t[0]
