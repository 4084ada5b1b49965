"""The tuner's cache tells apart live sets for which a knob acts and for which it does not: the contact pass's
block on both sides of 81,920 particles, the search order with and without a segment of more than 131,072; and
a knob that does nothing keeps its value. gather_block in sets where it acts gives the same results."""
import numpy as np
import pytest

from velvet_amd import scenes as S
from velvet_amd.solver import ClothSolver

pytestmark = pytest.mark.gpu


def _solver(sides, substeps=2):
    s = ClothSolver()
    for k, n in enumerate(sides):
        c = S.grid_cloth(n, 0.05, center=(0.0, 1.0, 0.0), jitter=2e-3, seed=k, stream=18)
        c.x[:, 1] += (0.04 * np.floor(3.0 * S.uniform(k, 19, c.n))).astype(np.float32)
        c.x[:, 0] *= np.float32(0.6)
        p = S.Params(num_substeps=substeps, num_iterations=2, friction=0.3, max_num_neighbors=30)
        s.load_scene(S.Scene(S.finish_params(p, [c]), [c], [S.sphere((0.1, 0.9, 0.05), 0.08)], 2))
    return s


@pytest.mark.parametrize("first,second", [((270,), (300,)), ((316, 316, 316), (450, 220, 220))])
def test_classes(first, second):
    """Both of one size class and segment class."""
    print(f"[gpu] tuned {first}, then {second}", flush=True)
    with _solver(first) as s:
        s.autotune(frames=2)
    with _solver(second) as s:
        assert s.autotune(frames=2, use_cache=True)["frame_ms"] > 0


def test_knob_without_effect_keeps_its_value():
    for block in (64, 128, 256):
        with _solver((100, 80), substeps=3) as s:
            s.set_tuning(gather_block=block)
            assert s.autotune(frames=1)["gather_block"] == block


def test_blocks_of_the_contact_pass_bit_identical():
    """More than 81,920 particles, so that the block acts; against eight neighbours at a time in smaller sets."""
    def run(sides, **tuning):
        with _solver(sides) as s:
            s.set_tuning(**tuning)
            for _ in range(2):
                s.Simulate()
            s.synchronize()
            return [(s.positions(k), s.velocities(k)) for k in range(len(sides))]

    sides = (257, 130, 33)
    want = [run(sides[:1])[0]]
    assert sum(n * n for n in sides) > 81920
    for block in (64, 128, 256):
        print(f"[gpu] contact pass in blocks of {block}", flush=True)
        got = run(sides, gather_block=block)
        want += got[len(want):]
        for (x, v), (xr, vr) in zip(got, want):
            assert np.isfinite(x).all() and np.array_equal(x, xr) and np.array_equal(v, vr)
