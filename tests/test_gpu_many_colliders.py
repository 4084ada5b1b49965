"""Updates of many colliders between frames: the same as with a wait in between on both sides of the count from
which they are copied, and an update of 256 takes at most three times one of 16 (one copy of 1.6 times the
time; in launches of eight it took eight times)."""
import time

import numpy as np
import pytest

from tests.test_gpu_frame_updates import _run
from velvet_amd import scenes as S
from velvet_amd._lib import check, lib
from velvet_amd.solver import ClothSolver, to_vtx_colliders

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count,graph,streams", [(32, True, 1), (33, False, 2), (70, True, 1)])
def test_updates_between_frames(count, graph, streams):
    print(f"[gpu] updates between frames, {count} colliders graph={graph} streams={streams}", flush=True)
    for (x, v), (xr, vr) in zip(_run(count, False, graph, streams), _run(count, True, False, 1)):
        assert np.isfinite(x).all() and np.array_equal(x, xr) and np.array_equal(v, vr)


def test_time_of_an_update():
    t = []
    for n in (16, 256):
        with ClothSolver() as s:
            c = S.grid_cloth(20, 0.05, center=(0.0, 1.0, 0.0))
            cols = [S.sphere((0.01 * k, 0.1, 0.0), 0.05) for k in range(n)]
            p = S.Params(num_substeps=1, num_iterations=1, enable_self_collision=False)
            s.load_scene(S.Scene(S.finish_params(p, [c]), [c], cols, 1))
            a = to_vtx_colliders(cols)
            s.Simulate()
            s.synchronize()
            best = np.inf
            for _ in range(6):
                b = time.perf_counter()
                for _ in range(30):
                    check(lib().vtx_set_colliders(s.h, 0, a, n))
                    s.synchronize()
                best = min(best, (time.perf_counter() - b) / 30)
            t.append(best)
    print(f"[gpu] updates of 16 and 256 colliders: {t[0] * 1e6:.1f} and {t[1] * 1e6:.1f} us", flush=True)
    assert t[1] < 3 * t[0]
