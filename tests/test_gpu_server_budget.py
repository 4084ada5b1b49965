"""What a job needs of a server's memory budget is what it registers: the same whether its dense attachments
are stored tile by tile or, where the budget asks, slot by slot, and however many tiles hold a bend. A job is
accepted at that size and rejected one byte below, and moves alike in either layout."""
import numpy as np
import pytest

from velvet_amd import scenes as S
from velvet_amd.server import DONE, REJECTED, Server

pytestmark = pytest.mark.gpu


def _scene(n, slots, general):
    cloths = [S.grid_cloth(n, 0.05, center=(0.0, 1.0, 0.0), jitter=2e-3, seed=n, stream=3, attached=tuple(range(slots)))]
    if general:
        cloths.append(S.grid_cloth(6, 0.05, center=(0.0, 2.0, 0.0)))
    p = S.Params(num_substeps=1, num_iterations=1)
    return S.Scene(S.finish_params(p, cloths), cloths, [], 3)


def _result(scene, budget):
    with Server(hbm_budget_bytes=budget) as sv:
        job = sv.submit(scene)
        if sv.status(job)[0] == REJECTED:
            return None
        for _ in range(5):
            sv.step()
        sv.drain()
        assert sv.status(job)[0] == DONE
        return sv.result(job)


@pytest.mark.parametrize("n,slots,general,needs", [(33, 33, 0, 497112), (100, 100, 0, 7241600), (129, 40, 0, 8054884),
                                                   (40, 8, 0, 569728), (17, 3, 0, 97152), (31, 0, 1, 545992), (48, 2, 1, 1346664)])
def test_budget_of_a_job(n, slots, general, needs):
    print(f"[gpu] budget n={n} slots={slots} general={general}", flush=True)
    scene = _scene(n, slots, general)
    assert _result(scene, needs - 1) is None
    x = _result(scene, needs)
    assert x is not None and np.isfinite(x).all() and np.array_equal(x, _result(scene, 1 << 30))
