"""Listed attachments on the general Jacobi path, four in flight: bit for bit the dense form's sums, at the edges of
a group of four and of the parts, with particles that have fewer of them; and eight of them take no more than a
quarter of a pass with bends (in flight 0.14 by their bytes and latency; one after another they took 0.34)."""
import dataclasses
import time

import numpy as np
import pytest

from velvet_amd import scenes as S
from velvet_amd.solver import ClothSolver

pytestmark = pytest.mark.gpu


def _cloth(n, bends, slots, seed=1):
    return S.grid_cloth(n, 0.05, center=(0.0, 1.0, 0.0), jitter=2e-3, seed=seed, stream=5, attached=tuple(range(slots)), bend_mode=bends)


def _listed(c, keep=None):
    o = np.lexsort((c.attach_slot, c.attach_pid))
    if keep is not None:
        o = o[keep[o]]
    return dataclasses.replace(c, attach_pid=c.attach_pid[o], attach_slot=c.attach_slot[o], attach_dist=c.attach_dist[o])


def _run(c, iterations=4, rounds=0):
    p = S.Params(num_substeps=2, num_iterations=iterations, enable_self_collision=False, long_range_stretchiness=0.97)
    with ClothSolver(stencil=False) as s:
        s.load_scene(S.Scene(S.finish_params(p, [c]), [c], [], 2))
        for _ in range(3):
            s.Simulate()
        s.synchronize()
        best = np.inf
        for _ in range(rounds):
            t = time.perf_counter()
            for _ in range(5):
                s.Simulate()
            s.synchronize()
            best = min(best, (time.perf_counter() - t) / 5)
        return best, s.positions(), s.velocities()


@pytest.mark.parametrize("n,bends,slots", [(2, "none", 1), (16, "pairs", 3), (17, "none", 4), (17, "pairs", 5), (20, "pairs", 8),
                                           (20, "none", 9), (33, "pairs", 17), (263, "pairs", 6), (263, "none", 13)])
@pytest.mark.parametrize("some", [False, True])
def test_listed_as_dense(n, bends, slots, some):
    """some: about half of the attachments, the others with a distance that is never exceeded in the dense form."""
    print(f"[gpu] n={n} bends={bends} slots={slots} some={some}", flush=True)
    c = _cloth(n, bends, slots)
    keep = S.uniform(n, 7, c.attach_pid.size) < 0.5 if some else np.ones(c.attach_pid.size, bool)
    keep[0] = True
    dense = dataclasses.replace(c, attach_dist=np.where(keep, c.attach_dist, np.float32(1e6)))
    _, x, v = _run(dense)
    _, xl, vl = _run(_listed(c, keep))
    assert np.isfinite(x).all() and np.array_equal(x, xl) and np.array_equal(v, vl)


def test_time_of_listed_attachments():
    t0, t8 = (_run(_listed(_cloth(600, "pairs", slots)) if slots else _cloth(600, "pairs", 0), 20, rounds=5)[0] for slots in (0, 8))
    print(f"[gpu] 360,000 particles, 40 passes: {t0 * 1e6:.0f} us without, {t8 * 1e6:.0f} us with 8 listed", flush=True)
    assert t8 < 1.25 * t0
