"""Fused Jacobi passes (several per launch, small and medium grid cloths) bit for bit against one pass per
launch: the same attachments listed particle by particle keep a cloth off the fused path, and sum alike.
Sides at the edges of the tiles (8, 12, 16) and around the tile counts where the side changes, pass counts
that split evenly and not, missing bending types, rest angles, and live sets that mix both kinds."""
import numpy as np
import pytest

from velvet_amd import scenes as S
from velvet_amd.solver import ClothSolver

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"[gpu] {msg}", flush=True)


def _cloth(n, bends, rest, seed):
    c = S.grid_cloth(n, 0.05, center=(0.0, 1.0, 0.0), jitter=2e-3, seed=seed, stream=9, attached=(0, n - 1),
                     bend_mode=bends)
    if rest:
        c.bend_rest = S.uniform(seed, 10, c.bend_rest.size, 0.0, 0.3).astype(np.float32)
    return c


def _listed(c):
    """The cloth with its attachments in particle-major order: stored as lists, one pass per launch."""
    o = np.lexsort((c.attach_slot, c.attach_pid))
    return S.Cloth(**{**c.__dict__, "attach_pid": c.attach_pid[o], "attach_slot": c.attach_slot[o],
                      "attach_dist": c.attach_dist[o]})


def _scene(c, iterations, substeps=2):
    p = S.Params(num_substeps=substeps, num_iterations=iterations, relaxation_factor=1.2)
    return S.Scene(S.finish_params(p, [c]), [c], [S.sphere((0.1, 0.8, 0.0), 0.15)], 3)


def _run(scenes, frames=3):
    with ClothSolver() as s:
        segs = [s.load_scene(sc) for sc in scenes]
        for _ in range(frames):
            s.Simulate()
        s.synchronize()
        return [(s.positions(k), s.velocities(k)) for k in segs]


@pytest.mark.parametrize("n,iterations,bends,rest", [
    (2, 3, "pairs", False), (3, 4, "pairs", False), (8, 1, "pairs", False), (9, 2, "quad", False),
    (16, 5, "pairs", True), (25, 7, "none", False), (41, 10, "pairs", True),                    # side 8
    (96, 10, "pairs", False), (133, 4, "quad", True), (192, 5, "pairs", False),                 # side 12
    (193, 7, "pairs", False), (224, 2, "pairs", True), (225, 3, "pairs", False),                # side 16, then none
])
def test_fused_equals_single_passes(n, iterations, bends, rest):
    say(f"fused passes n={n} iterations={iterations} bends={bends} rest={rest}")
    c = _cloth(n, bends, rest, seed=n)
    (xa, va), = _run([_scene(c, iterations)])
    (xb, vb), = _run([_scene(_listed(c), iterations)])
    assert np.isfinite(xa).all() and np.array_equal(xa, xb) and np.array_equal(va, vb)


@pytest.mark.parametrize("iterations", [1, 2, 4, 5, 10])
def test_fused_and_single_cloths_in_one_solver(iterations):
    """Both kinds leave a substep in the same ping-pong buffer whatever the pass count."""
    say(f"fused and single passes together, iterations={iterations}")
    scenes = [_scene(_cloth(20, "pairs", False, 1), iterations), _scene(_listed(_cloth(17, "pairs", False, 2)), iterations),
              _scene(_cloth(33, "quad", True, 3), iterations)]
    mixed = _run(scenes)
    for sc, (x, v) in zip(scenes, mixed):
        (xa, va), = _run([sc])
        assert np.array_equal(x, xa) and np.array_equal(v, va)
