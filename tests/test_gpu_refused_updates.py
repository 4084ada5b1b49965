"""A collider or slot update refused because the caller's stream is being captured changes nothing: neither
the frames that follow nor what a later upload of the segment takes from the host."""
import ctypes as C

import numpy as np
import pytest

from velvet_amd import scenes as S
from velvet_amd.solver import ClothSolver

pytestmark = pytest.mark.gpu


def _run(refused):
    hip = C.CDLL("libamdhip64.so")
    stream, graph = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreate(C.byref(stream)) == 0
    c = S.grid_cloth(20, 0.05, center=(0.0, 1.0, 0.0), jitter=2e-3, seed=1, stream=17, attached=(0, 19))
    p = S.finish_params(S.Params(num_substeps=2, num_iterations=3), [c])
    try:
        with ClothSolver(use_graph=False) as s:
            s.load_scene(S.Scene(p, [c], [S.sphere((0.1, 0.8, 0.0), 0.15)], 2))
            s.set_stream(stream.value)
            s.Simulate()
            s.synchronize()
            if refused:
                assert hip.hipStreamBeginCapture(stream, 1) == 0          # thread-local mode
                try:
                    with pytest.raises(Exception):
                        s.UpdateColliders([S.sphere((0.1, 0.9, 0.0), 0.2)])
                    with pytest.raises(Exception):
                        s.SetAttachSlotPosition(0, c.slots[0] + np.float32([0.0, 0.1, 0.0]))
                finally:
                    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
                    hip.hipGraphDestroy(graph)
            s.Simulate()
            s.set_params(p)                                               # the segment is packed and uploaded again
            s.Simulate()
            s.synchronize()
            out = s.positions(), s.velocities()
            s.set_stream(None)
            return out
    finally:
        hip.hipStreamDestroy(stream)


def test_refused_updates_change_nothing():
    print("[gpu] updates during a capture", flush=True)
    for got, want in zip(_run(True), _run(False)):
        assert np.isfinite(got).all() and np.array_equal(got, want)
