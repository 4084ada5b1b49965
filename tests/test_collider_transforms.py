"""Collider matrices as the solver passes them equal scenes.collider_matrices bit for bit, with the rotation
zero (no matrix products) and not, finite and not."""
import numpy as np
import pytest

from velvet_amd import scenes as S
from velvet_amd.solver import to_vtx_colliders


@pytest.mark.parametrize("position,scale,rotation", [
    ((0.1, -0.7, 1 / 3), (0.6, 0.6, 0.6), (0.0, 0.0, 0.0)), ((-0.0, 0.0, 1e30), (1e-30, -2.0, 3.0), (0, 0, -0.0)),
    ((0.1, 0.2, 0.3), (1.0, 2.0, 3.0), (10.0, -20.0, 400.0)), ((float("inf"), 0.0, 0.0), (1.0, 1.0, 1.0), (0.0, 0.0, 0.0)),
    (np.float32([0.1, 0.2, 0.3]), np.float32([1, 2, 3]), np.zeros(3, np.float32)),
])
def test_transforms(position, scale, rotation):
    c = S.Collider(S.SPHERE, position, scale, rotation, last_position=(0.3, 0.2, 0.1))
    a = to_vtx_colliders([c])[0]
    cur, last = S.collider_matrices(c)
    assert np.array_equal(np.array(a.cur[:], np.float32), cur, equal_nan=True)
    assert np.array_equal(np.array(a.last[:], np.float32), last, equal_nan=True)
