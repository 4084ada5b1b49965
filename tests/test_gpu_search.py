"""The neighbour search at the edges of its waves, runs and candidate chunks, bit-exact against the
binary32 restatement: object counts around the particles of a wave, runs of one cell longer than a
wave's particles, candidate totals around one and two chunks of 64, and the count where a wave starts
to take 32 particles instead of 8."""
import numpy as np
import pytest

from tests.test_gpu_hash_objects import check_against_restatement, hash_objects, say
from velvet_amd import scenes as S

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.mark.parametrize("n,per_cell,M,K", [
    (1, 1, 2, 64), (7, 3, 14, 64), (8, 3, 16, 64), (9, 9, 18, 64), (33, 40, 66, 64),    # waves of 8, one run
    (257, 2, 514, 64), (257, 2.4, 514, 5), (300, 2.4, 97, 64),                          # about 64 candidates
    (1000, 4.7, 2000, 64), (1000, 5, 2000, 63), (1000, 30, 1, 64),                      # about 128, full lists, one bucket
    ((1 << 17), 3, 1 << 18, 64), ((1 << 17) + 1, 3, 1 << 18, 64), ((1 << 17) + 33, 5, 400_003, 61),
])
def test_search_edges(n, per_cell, M, K):
    say(f"search n={n} per cell {per_cell} M={M} K={K}")
    cell, diameter = F32(0.1), F32(0.06)
    side = max((n / per_cell) ** (1 / 3), 1.0) * float(cell)          # per_cell objects in a cell on average
    p = S.uniform(n, 1, 3 * n, -0.4 * side, 0.6 * side).reshape(n, 3).astype(F32)
    x0 = S.uniform(n, 2, 3 * n, 0.0, 4 * side).reshape(n, 3).astype(F32)
    check_against_restatement(hash_objects(p, x0, cell, diameter, M, K), p, x0, cell, diameter, M, K)
