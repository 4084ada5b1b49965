"""The hash build by cell ranges where cells are crowded: bit-exact against the binary32 restatement and the
device-wide sort for ranges sorted in LDS, ranges that hold more than their list, more crowded cells than
one run takes, everything in one cell and tables smaller than the limit; and no more than three times the
time of evenly filled cells (a sort of at most 4,096 words on top of the build; a run over all keys for each
crowded cell took five to ten times)."""
import ctypes as C
import time

import numpy as np
import pytest

from tests.hipmem import DeviceArray, hip
from tests.test_gpu_hash_objects import check_against_restatement, hash_objects, say
from velvet_amd import scenes as S
from velvet_amd._lib import VtxHashParams, check, lib
from velvet_amd.solver import ClothSolver

pytestmark = pytest.mark.gpu
F32 = np.float32
CELL, DIAMETER = F32(0.1), F32(0.06)


def _cells(at, n, seed):
    """n objects dealt to the cells `at` in turn."""
    p = (at[np.arange(n) % len(at)] + S.uniform(seed, 3, 3 * n, 0.1, 0.9).reshape(n, 3)) * 0.1
    return p.astype(F32), S.uniform(seed, 2, 3 * n, 0.0, 4.0).reshape(n, 3).astype(F32)


def _block(count):
    e = int(np.ceil(count ** (1 / 3)))
    return np.stack(np.meshgrid(*[np.arange(e)] * 3, indexing="ij"), -1).reshape(-1, 3)[:count]


def _first_range(count, n, M):
    """Cells whose hashes fall in the first range of the table."""
    width = -(-M // max(-(-n // 1024), -(-M // 4096)))
    at = np.stack(np.meshgrid(*[np.arange(-60, 60)] * 3, indexing="ij"), -1).reshape(-1, 3)
    u = at.astype(np.int32).astype(np.uint32)
    h = ((u[:, 0] * np.uint32(92837111)) ^ (u[:, 1] * np.uint32(689287499)) ^ (u[:, 2] * np.uint32(283923481))).view(np.int32)
    at = at[np.abs(h.astype(np.int64)) % M < width]
    assert len(at) >= count
    return at[:count]


@pytest.mark.parametrize("n,M,cells", [
    (4096, 8192, 8), (8192, 16384, 30), (8192, 16384, 1), (8193, 16386, 31), (20000, 150, 8000), (131072, 1000, 40000),
    (131072, 262144, 60), (131072, 262144, 1), (131072, 64, 40000), (131072, 63, 40000), (5000, 2, 3), (5000, 3, 3),
])
def test_crowded_tables(n, M, cells):
    say(f"crowded hash n={n} M={M} cells={cells}")
    p, x0 = _cells(_block(cells), n, n)
    check_against_restatement(hash_objects(p, x0, CELL, DIAMETER, M, 4), p, x0, CELL, DIAMETER, M, 4)


@pytest.mark.parametrize("n,cells", [(4096, 15), (4097, 15), (8192, 40), (8193, 40), (131072, 255), (131072, 257), (131072, 500)])
def test_crowded_cells_of_one_range(n, cells):
    say(f"crowded hash, one range, n={n} cells={cells}")
    M = 2 * n
    p, x0 = _cells(_first_range(cells, n, M), n, n)
    check_against_restatement(hash_objects(p, x0, CELL, DIAMETER, M, 4), p, x0, CELL, DIAMETER, M, 4)


@pytest.mark.parametrize("sides,squeeze", [((90,), 0.02), ((200, 150), 0.02), ((362,), 0.0), ((300,) * 3, 0.05), ((300,) * 3, 0.0)])
def test_crowded_segments_same_as_device_wide_sort(sides, squeeze):
    say(f"crowded segments {sides} squeezed to {squeeze}")
    out = []
    for on in (1, 0):
        with ClothSolver(use_graph=False) as s:
            for k, n in enumerate(sides):
                c = S.grid_cloth(n, 0.05, center=(0.0, 1.0, 0.0), jitter=2e-3, seed=k, stream=16)
                c.x[:, ::2] *= F32(squeeze)
                s.load_scene(S.Scene(S.finish_params(S.Params(num_substeps=2, num_iterations=1), [c]), [c], [], 2))
            s.set_tuning(hash_lds=on)
            s.run_hash()
            out.append([s.read_hash(k) for k in range(len(sides))])
    for a, b in zip(*out):
        for x, y in zip(a[:-1], b[:-1]):
            assert np.array_equal(x, y)
        live = [np.cumprod(t[-1] != 0xFFFFFFFF, axis=0).astype(bool) for t in (a, b)]   # up to the sentinel
        assert np.array_equal(*live) and np.array_equal(a[-1][live[0]], b[-1][live[0]])


def _time(p, x0, M, K=4):
    n = len(p)
    prm = VtxHashParams(num_objects=n, max_num_neighbors=K, cell_spacing=CELL, cell_spacing2=F32(CELL * CELL), table_size=M,
                        particle_diameter2=F32(DIAMETER * DIAMETER))
    arrays = [DeviceArray(shape=(k,), dtype=np.uint32) for k in (n, n, M, M, K * n)] + [DeviceArray(p), DeviceArray(x0)]
    best = np.inf
    for _ in range(6):
        hip().hipDeviceSynchronize()
        t = time.perf_counter()
        for _ in range(20):
            check(lib().vtx_hash_objects(*[a.ptr for a in arrays], C.byref(prm), None))
        hip().hipDeviceSynchronize()
        best = min(best, (time.perf_counter() - t) / 20)
    return best


@pytest.mark.parametrize("n,even,crowded", [(131072, (262144, 1311), (262144, 937)), (131072, (4000, 40000), (1000, 40000)),
                                            (65536, (131072, 656), (131072, 469))])
def test_time_of_crowded_cells(n, even, crowded):
    """Cells of 100 against 140 objects, and a table four times as crowded."""
    t = [_time(*_cells(_block(cells), n, 1), M) for M, cells in (even, crowded)]
    say(f"crowded hash n={n}: {t[0] * 1e6:.1f} us evenly filled, {t[1] * 1e6:.1f} us crowded")
    assert t[1] < 3 * t[0]
