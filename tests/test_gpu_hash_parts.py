"""The hash build by cell ranges at its edges, bit-exact against the binary32 restatement: object counts
where the keys move to a kernel of their own and where the device-wide sort takes over, table sizes around
the width of a range, cells around the size that is placed by a run over the keys, and ranges that hold more
particles than their list in LDS."""
import numpy as np
import pytest

from tests.test_gpu_hash_objects import check_against_restatement, hash_objects, say
from velvet_amd import scenes as S
from velvet_amd.solver import ClothSolver

pytestmark = pytest.mark.gpu
F32 = np.float32


def _check(p, x0, M, K):
    cell, diameter = F32(0.1), F32(0.06)
    check_against_restatement(hash_objects(p, x0, cell, diameter, M, K), p, x0, cell, diameter, M, K)


def _objects(n, side):
    p = S.uniform(n, 1, 3 * n, -0.4 * side, 0.6 * side).reshape(n, 3).astype(F32)
    return p, S.uniform(n, 2, 3 * n, 0.0, 4 * side).reshape(n, 3).astype(F32)


@pytest.mark.parametrize("n,M", [
    (1, 1), (63, 4095), (1023, 4096), (1024, 4097), (1025, 524288), (1025, 524289), (5000, 9999),
    (8191, 16382), (8192, 16384), (8193, 16386), (16385, 4096), (24577, 3), (40001, 30011), (131072, 262144), (131073, 262146),
])
def test_counts_and_table_sizes(n, M):
    say(f"hash ranges n={n} M={M}")
    _check(*_objects(n, max((n / 2.5) ** (1 / 3), 1.0) * 0.1), M, 8)


@pytest.mark.parametrize("n,per", [(1032, 128), (1032, 129), (4096, 64), (4160, 64), (9216, 96), (9100, 130), (20000, 2500)])
def test_crowded_cells_in_one_range(n, per):
    """Cells of `per` objects (indices interleaved) whose hashes all fall in the first range of the table."""
    say(f"hash ranges n={n}, cells of {per}")
    M = 8 * n
    width = -(-M // max(-(-n // 1024), -(-M // 4096)))
    at = np.stack(np.meshgrid(*[np.arange(-60, 60)] * 3, indexing="ij"), -1).reshape(-1, 3)
    u = at.astype(np.int32).astype(np.uint32)
    h = ((u[:, 0] * np.uint32(92837111)) ^ (u[:, 1] * np.uint32(689287499)) ^ (u[:, 2] * np.uint32(283923481))).view(np.int32)
    at = at[np.abs(h.astype(np.int64)) % M < width]
    cells = -(-n // per)
    assert len(at) >= cells
    p, x0 = _objects(n, 1.0)
    p = ((at[np.arange(n) % cells] + S.uniform(n, 3, 3 * n, 0.1, 0.9).reshape(n, 3)) * 0.1).astype(F32)
    _check(p, x0, M, 4)


@pytest.mark.parametrize("n", [8000, 20000, 140000])
def test_positions_on_cell_faces(n):
    """Coordinates at and one to three steps off multiples of the cell size, up to 2^28 cells out, and tiny ones."""
    say(f"hash of positions on cell faces n={n}")
    cell = F32(0.1)
    far = np.exp2(S.uniform(n, 4, 3 * n, 0.0, 28.0)) * np.where(S.uniform(n, 5, 3 * n) < 0.5, -1.0, 1.0)
    p = (np.floor(far).astype(F32) * cell).view(np.int32) + np.floor(S.uniform(n, 6, 3 * n, -3.0, 4.0)).astype(np.int32)
    p = p.view(F32).reshape(n, 3).copy()
    p[::7] = (S.uniform(n, 7, 3 * len(p[::7]), -4.0, 4.0).reshape(-1, 3) * F32(1e-39)).astype(F32)
    p[::11, 0] = 0.0
    p[::13, 1] = -0.0
    _check(p, S.uniform(n, 2, 3 * n, 0.0, 1e3).reshape(n, 3).astype(F32), 2 * n - 1, 2)


@pytest.mark.parametrize("sides", [(31, 32, 33), (90, 91), (64, 150, 363), (128,) * 17])
def test_segments_same_as_device_wide_sort(sides):
    """Frames of self-colliding cloths with the build by ranges and by the device-wide sort."""
    say(f"hash ranges, segments {sides}")
    out = []
    for on in (1, 0):
        with ClothSolver(use_graph=False) as s:
            for k, n in enumerate(sides):
                c = S.grid_cloth(n, 0.05, center=(0.0, 1.0, 0.0), jitter=2e-3, seed=k, stream=16)
                c.x[:, 1] = (1.0 + 0.05 * np.abs(np.sin(40.0 * c.x[:, 0]))).astype(F32)
                s.load_scene(S.Scene(S.finish_params(S.Params(num_substeps=2, num_iterations=2), [c]), [c], [], 2))
            s.set_tuning(hash_lds=on)
            for _ in range(2):
                s.Simulate()
            s.synchronize()
            out.append([(s.positions(k), s.velocities(k), *s.read_hash(k)) for k in range(len(sides))])
    for a, b in zip(*out):
        for x, y in zip(a[:-1], b[:-1]):
            assert np.array_equal(x, y)
        live = [np.cumprod(t[-1] != 0xFFFFFFFF, axis=0).astype(bool) for t in (a, b)]   # up to the sentinel
        assert np.array_equal(*live) and np.array_equal(a[-1][live[0]], b[-1][live[0]])
