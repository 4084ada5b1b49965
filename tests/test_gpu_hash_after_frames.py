"""vtx_run_hash after frames, without positions of the caller's: the tables of fused Jacobi passes equal those of
one pass per launch (the same attachments listed particle by particle) bit for bit, for pass counts that split
evenly and not, with and without a contact pass, in sets of one kind and mixed, on one and several streams, and
beside a segment whose positions the caller wrote."""
import numpy as np
import pytest

from velvet_amd import scenes as S
from velvet_amd.solver import ClothSolver

pytestmark = pytest.mark.gpu


def _cloth(n, listed, seed):
    c = S.grid_cloth(n, 0.05, center=(0.0, 1.0, 0.0), jitter=4e-3, seed=seed, stream=9, attached=(0, n - 1))
    c.x[:, 1] += (0.08 * np.abs(np.sin(9.0 * c.x[:, 0]))).astype(np.float32)
    if listed:
        o = np.lexsort((c.attach_slot, c.attach_pid))
        c.attach_pid, c.attach_slot, c.attach_dist = c.attach_pid[o], c.attach_slot[o], c.attach_dist[o]
    return c


def _hashes(sides, listed, substeps, iterations, graph=True, streams=1, write=False):
    with ClothSolver(use_graph=graph) as s:
        segs = []
        for k, n in enumerate(sides):
            c = _cloth(n, listed, k)
            p = S.Params(num_substeps=substeps, num_iterations=iterations)
            segs.append(s.load_scene(S.Scene(S.finish_params(p, [c]), [c], [S.sphere((0.1, 0.9, 0.0), 0.15)], 2)))
        s.set_tuning(streams=streams)
        out = []
        for f in range(2):
            s.Simulate()
            if write and f:
                s.write_predicted(_cloth(sides[-1], False, 7).x, seg=segs[-1])
            s.run_hash()
            for k in segs:
                t = s.read_hash(k)
                live = np.cumprod(t[-1] != 0xFFFFFFFF, axis=0).astype(bool)
                out.append([*t[:-1], live, np.where(live, t[-1], 0)])
        return out


@pytest.mark.parametrize("sides,substeps,iterations,graph,streams,write", [
    ((20,), 1, 1, True, 1, False), ((20,), 1, 2, True, 1, False), ((20,), 2, 3, True, 1, False), ((20,), 3, 4, False, 1, False),
    ((41,), 2, 5, True, 1, True), ((41,), 5, 10, True, 1, False), ((130,), 2, 7, True, 1, False), ((193,), 2, 4, False, 1, False),
    ((193,), 3, 5, True, 1, False), ((20, 33, 48), 2, 6, False, 2, True), ((20, 33, 48), 3, 10, True, 3, True),
])
def test_fused_equals_single_passes(sides, substeps, iterations, graph, streams, write):
    print(f"[gpu] hash after frames {sides} {substeps} x {iterations}", flush=True)
    got = _hashes(sides, False, substeps, iterations, graph, streams, write)
    want = _hashes(sides, True, substeps, iterations, graph, streams, write)
    for a, b in zip(got, want):
        for x, y in zip(a, b):
            assert np.array_equal(x, y)
