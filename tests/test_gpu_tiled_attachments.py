"""Grid cloths with 32 or more dense attachment slots (targets tiled, four slots to a vector, slots split
over four threads) bit for bit against the same attachments listed particle by particle: slot counts at the
threshold and around multiples of four and of the four shares, tiles cut off at the cloth's edge, distances of
zero, both batch depths, every bending form."""
import numpy as np
import pytest

from velvet_amd import scenes as S
from velvet_amd.solver import ClothSolver

pytestmark = pytest.mark.gpu


def _run(c, iterations, **tuning):
    p = S.Params(num_substeps=2, num_iterations=iterations, enable_self_collision=False, relaxation_factor=1.1,
                 long_range_stretchiness=1.05)
    sc = S.Scene(S.finish_params(p, [c]), [c], [S.sphere((0.1, 0.9, 0.05), 0.08)], 2)
    with ClothSolver() as s:
        s.load_scene(sc)
        s.set_tuning(**tuning)
        for _ in range(2):
            s.Simulate()
        s.synchronize()
        return s.positions(), s.velocities()


@pytest.mark.parametrize("n,slots,bends,rest", [
    (8, 32, "pairs", False), (16, 31, "pairs", False), (16, 32, "quad", False), (17, 33, "pairs", True),
    (33, 34, "none", False), (33, 35, "pairs", False), (40, 61, "quad", True), (47, 64, "pairs", False),
    (31, 66, "pairs", True), (17, 1100, "pairs", False),   # the last: slot-major, tiles would store 3.5 times as much
])
def test_tiled_equals_listed(n, slots, bends, rest):
    print(f"[gpu] tiled attachments n={n} slots={slots} bends={bends} rest={rest}", flush=True)
    pick = np.resize(np.argsort(S.uniform(n, 14, n * n)), slots)
    c = S.grid_cloth(n, 0.05, center=(0.0, 1.0, 0.0), jitter=2e-3, seed=n, stream=13,
                     attached=tuple(int(i) for i in pick), bend_mode=bends)
    if rest:
        c.bend_rest = S.uniform(n, 10, c.bend_rest.size, 0.0, 0.3).astype(np.float32)
    u = S.uniform(n, 15, c.attach_dist.size)
    c.attach_dist = np.where(u < 0.1, 0.0, np.where(u < 0.6, 0.5 * c.attach_dist, c.attach_dist)).astype(np.float32)
    o = np.lexsort((c.attach_slot, c.attach_pid))
    listed = S.Cloth(**{**c.__dict__, "attach_pid": c.attach_pid[o], "attach_slot": c.attach_slot[o],
                        "attach_dist": c.attach_dist[o]})
    want = _run(listed, 3)
    assert np.isfinite(want[0]).all()
    for batch in (4, 16, 64):
        for a, b in zip(_run(c, 3, lra_batch=batch), want):
            assert np.array_equal(a, b), batch
