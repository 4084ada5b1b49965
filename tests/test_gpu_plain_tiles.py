"""General-path tiles without bending constraints: bit for bit alike in a launch of their own and along with
tiles that have bends, at tile edges and on both sides of the count where they get one, with listed and dense
attachments; and a pass over them takes no more than 0.27 of a pass with three bends a particle (one thread
per particle 0.20 by its share of the loads; the workgroups of the bends' evaluation took 0.33)."""
import time

import numpy as np
import pytest

from velvet_amd import scenes as S
from velvet_amd.solver import ClothSolver

pytestmark = pytest.mark.gpu


def _scene(n, bends, slots, seed, selfcol=True):
    c = S.grid_cloth(n, 0.05, center=(0.0, 1.0, 0.0), jitter=2e-3, seed=seed, stream=9, attached=tuple(range(slots)), bend_mode=bends)
    if slots == 3:                                             # particle by particle: listed
        o = np.lexsort((c.attach_slot, c.attach_pid))
        c.attach_pid, c.attach_slot, c.attach_dist = c.attach_pid[o], c.attach_slot[o], c.attach_dist[o]
    p = S.Params(num_substeps=2, num_iterations=3, enable_self_collision=selfcol)
    return S.Scene(S.finish_params(p, [c]), [c], [S.sphere((0.1, 0.8, 0.0), 0.15)], 2)


def _run(scenes, streams=1):
    with ClothSolver(stencil=False) as s:
        segs = [s.load_scene(sc) for sc in scenes]
        s.set_tuning(streams=streams)
        for _ in range(2):
            s.Simulate()
        s.synchronize()
        return [(s.positions(k), s.velocities(k), s.normals(k)) for k in segs]


@pytest.mark.parametrize("sides,streams", [((2, 20), 1), ((16, 17), 1), ((255, 20), 1), ((257, 20), 1), ((300, 40, 33), 2), ((1027, 30), 1)])
def test_plain_tiles_beside_bent_ones(sides, streams):
    print(f"[gpu] plain tiles {sides} streams={streams}", flush=True)
    scenes = [_scene(n, "none" if k != 1 else "pairs", (2, 0, 3)[k], k) for k, n in enumerate(sides)]
    for sc, got in zip(scenes, _run(scenes, streams)):
        for a, b in zip(got, _run([sc])[0]):
            assert np.isfinite(a).all() and np.array_equal(a, b)


def test_time_of_plain_tiles():
    t = []
    for bends in ("none", "pairs"):
        with ClothSolver(stencil=False) as s:
            sc = _scene(700, bends, 0, 1, selfcol=False)
            sc.params.num_iterations = 20
            s.load_scene(sc)
            s.Simulate()
            s.synchronize()
            best = np.inf
            for _ in range(5):
                a = time.perf_counter()
                for _ in range(5):
                    s.Simulate()
                s.synchronize()
                best = min(best, (time.perf_counter() - a) / 5)
            t.append(best)
    print(f"[gpu] frames of 40 passes, 490,000 particles: {t[0] * 1e6:.0f} us without, {t[1] * 1e6:.0f} us with bending", flush=True)
    assert t[0] < 0.27 * t[1]
