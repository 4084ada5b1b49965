"""The general Jacobi path's bend records per tile: the same cloth with its particles renumbered at random
gives the same trajectories bit for bit. Renumbering keeps every particle's constraints and their order but
deals the particles to other tiles, so records, rounds and entries change: tiles whose records take one
round and several, particles with more bend entries than are staged, partial tiles, and a live set of more
tiles than CUs (one record a thread)."""
import dataclasses

import numpy as np
import pytest

from velvet_amd import scenes as S
from velvet_amd.solver import ClothSolver

pytestmark = pytest.mark.gpu


def _run(c, iterations):
    p = S.Params(num_substeps=2, num_iterations=iterations, enable_self_collision=False, relaxation_factor=1.3)
    sc = S.Scene(S.finish_params(p, [c]), [c], [S.sphere((0.1, 0.9, 0.05), 0.08)], 2)
    with ClothSolver(stencil=False) as s:
        s.load_scene(sc)
        for _ in range(2):
            s.Simulate()
        s.synchronize()
        return s.positions(), s.velocities(), s.normals()


@pytest.mark.parametrize("n,repeat,iterations", [(3, 1, 2), (16, 1, 3), (20, 1, 4), (20, 2, 4), (20, 3, 4), (17, 7, 3),
                                                 (40, 1, 3), (257, 1, 2), (260, 2, 2)])
def test_renumbered_particles_bit_identical(n, repeat, iterations):
    """Every bend registered `repeat` times: 1 to 7 times the records and entries."""
    print(f"[gpu] general path n={n} repeat={repeat}", flush=True)
    c = S.grid_cloth(n, 0.05, center=(0.0, 1.0, 0.0), jitter=2e-3, seed=n, stream=11, attached=(0, n - 1))
    rest = S.uniform(n, 12, c.bend_rest.size, 0.0, 0.2).astype(np.float32)
    c = dataclasses.replace(c, bend=np.repeat(c.bend, repeat, axis=0), bend_rest=np.repeat(rest, repeat))
    to = np.argsort(S.uniform(n, 13, c.n))                       # new number of particle i
    back = np.argsort(to)
    m = dataclasses.replace(c, x=c.x[back], tris=to[c.tris].astype(np.uint32), stretch=to[c.stretch].astype(np.int32),
                            bend=to[c.bend].astype(np.uint32),
                            attach_dist=c.attach_dist.reshape(2, c.n)[:, back].reshape(-1))
    for a, b in zip(_run(c, iterations), _run(m, iterations)):
        assert np.isfinite(a).all() and np.array_equal(a, b[to])
