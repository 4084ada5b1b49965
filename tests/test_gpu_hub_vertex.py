"""The general Jacobi path with a vertex of very many bends (a fan of triangles around it): the rounds over a
tile's bend records go on where they stopped, so the time grows with the bends (four times as many within six
times the time; every round over all entries took twelve times), and the particles' numbers don't matter."""
import dataclasses
import time

import numpy as np
import pytest

from velvet_amd import scenes as S
from velvet_amd.solver import ClothSolver

pytestmark = pytest.mark.gpu


def _fan(d, order=None):
    """d triangles around particle 0; order: new numbers of the particles."""
    a = np.linspace(0.0, 2.0 * np.pi, d, endpoint=False)
    x = np.zeros((d + 1, 3))
    x[1:, 0], x[1:, 2] = np.cos(a), np.sin(a)
    x[:, 1] = 1.0 + 0.01 * S.uniform(d, 1, d + 1)
    k = np.arange(d)
    tris = np.stack([np.zeros(d, int), 1 + k, 1 + (k + 1) % d], 1)
    c = S.mesh_cloth(x.astype(np.float32), tris.astype(np.uint32), 0.01)
    if order is not None:
        back = np.argsort(order)
        c.x, c.tris = c.x[back], order[c.tris].astype(np.uint32)
        c.stretch, c.bend = order[c.stretch].astype(np.int32), order[c.bend].astype(np.uint32)
    p = S.Params(num_substeps=2, num_iterations=4, enable_self_collision=False)
    return S.Scene(S.finish_params(p, [c]), [c], [], 2)


def _run(scene, frames=2, **kw):
    with ClothSolver(**kw) as s:
        s.load_scene(scene)
        s.Simulate()
        s.synchronize()
        t = time.perf_counter()
        for _ in range(frames):
            s.Simulate()
        s.synchronize()
        return (time.perf_counter() - t) / frames, s.positions(), s.velocities()


@pytest.mark.parametrize("d", [767, 1536, 1537, 6000])
def test_renumbered_fan(d):
    print(f"[gpu] fan of {d}", flush=True)
    to = np.argsort(S.uniform(d, 13, d + 1))
    _, x, v = _run(_fan(d))
    _, xr, vr = _run(_fan(d, to))
    assert np.isfinite(x).all() and np.array_equal(x, xr[to]) and np.array_equal(v, vr[to])


@pytest.mark.parametrize("n,repeat", [(20, 5), (20, 6), (262, 5), (262, 6)])
def test_renumbered_grid(n, repeat):
    """60 and 72 entries of a particle, on both sides of the count where rounds keep a particle's place, in sets of
    no more tiles than CUs and of more."""
    print(f"[gpu] grid of {n}, bends {repeat} times", flush=True)
    c = S.grid_cloth(n, 0.05, center=(0.0, 1.0, 0.0), jitter=2e-3, seed=n, stream=11)
    rest = S.uniform(n, 12, c.bend_rest.size, 0.0, 0.2).astype(np.float32)
    c.bend, c.bend_rest = np.repeat(c.bend, repeat, axis=0), np.repeat(rest, repeat)
    to = np.argsort(S.uniform(n, 13, c.n))
    m = dataclasses.replace(c, x=c.x[np.argsort(to)], tris=to[c.tris].astype(np.uint32), stretch=to[c.stretch].astype(np.int32),
                            bend=to[c.bend].astype(np.uint32))
    p = S.Params(num_substeps=2, num_iterations=2, enable_self_collision=False)
    (_, x, v), (_, xr, vr) = (_run(S.Scene(S.finish_params(p, [k]), [k], [], 2), stencil=False) for k in (c, m))
    assert np.isfinite(x).all() and np.array_equal(x, xr[to]) and np.array_equal(v, vr[to])


def test_time_grows_with_the_bends():
    t = [_run(_fan(d))[0] for d in (5000, 20000)]
    print(f"[gpu] fans of 5,000 and 20,000: {t[0] * 1e3:.1f} and {t[1] * 1e3:.1f} ms a frame", flush=True)
    assert t[1] < 6 * t[0]
