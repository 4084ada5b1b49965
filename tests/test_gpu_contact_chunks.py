"""The contact pass with eight neighbours at a time (small live sets) bit for bit against four (large ones):
the same cloths with and without a large bystander in the solver, lists of every length up to caps that are
and are not multiples of four and eight."""
import numpy as np
import pytest

from velvet_amd import scenes as S
from velvet_amd.solver import ClothSolver

pytestmark = pytest.mark.gpu


def _scene(n, cap, seed):
    c = S.grid_cloth(n, 0.05, center=(0.0, 1.0, 0.0), jitter=2e-3, seed=seed, stream=18)
    c.x[:, 1] += (0.04 * np.floor(3.0 * S.uniform(seed, 19, c.n))).astype(np.float32)
    c.x[:, 0] *= np.float32(0.6)
    p = S.Params(num_substeps=3, num_iterations=2, max_num_neighbors=cap, friction=0.3)
    return S.Scene(S.finish_params(p, [c]), [c], [S.sphere((0.1, 0.9, 0.05), 0.08)], 2)


def _run(scenes, bystander):
    with ClothSolver() as s:
        segs = [s.load_scene(sc) for sc in scenes]
        if bystander:
            c = S.grid_cloth(300, 0.05, center=(0.0, 50.0, 0.0))
            p = S.Params(num_substeps=3, num_iterations=2, enable_self_collision=False)
            s.load_scene(S.Scene(S.finish_params(p, [c]), [c], [], 2))
        for _ in range(2):
            s.Simulate()
        s.synchronize()
        return [(s.positions(k), s.velocities(k)) for k in segs]


@pytest.mark.parametrize("n,cap", [(2, 1), (17, 2), (24, 4), (24, 7), (24, 9), (24, 12), (40, 63), (257, 64)])
def test_eight_equal_four(n, cap):
    print(f"[gpu] contact chunks n={n} cap={cap}", flush=True)
    scenes = [_scene(n, cap, 1)] + ([_scene(33, 13, 2)] if n < 257 else [])
    for (x, v), (xr, vr) in zip(_run(scenes, False), _run(scenes, True)):
        assert np.isfinite(x).all() and np.array_equal(x, xr) and np.array_equal(v, vr)
