"""The search's stores on both sides of 2^22 objects, where the entries' byte offsets leave 32 bits: a small
cluster whose objects have the lowest and the highest indices among millions of lone ones has the lists it
has by itself."""
import numpy as np
import pytest

from tests.test_gpu_hash_objects import SENT, hash_objects, say
from velvet_amd import scenes as S

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.mark.parametrize("n", [(1 << 22) - 1, 1 << 22])
def test_cluster_among_lone_objects(n):
    say(f"search n={n}")
    cell, diameter, K, m = F32(0.1), F32(0.06), 32, 1000
    pc = S.uniform(m, 1, 3 * m, 0.0, 0.6).reshape(m, 3).astype(F32)
    xc = S.uniform(m, 2, 3 * m, 0.0, 4.0).reshape(m, 3).astype(F32)
    i = np.arange(n)
    p = (np.stack([i % 170, i // 170 % 170, i // (170 * 170)], 1) * 0.5 + 10.0).astype(F32)   # apart by five cells
    at = np.concatenate([np.arange(m // 2), np.arange(n - m // 2, n)])
    p[at] = pc
    x0 = p.copy()
    x0[at] = xc
    want = hash_objects(pc, xc, cell, diameter, 2 * n, K)[4]
    got = hash_objects(p, x0, cell, diameter, 2 * n, K)[4]
    live = np.cumprod(want != SENT, axis=0).astype(bool)
    assert live.any()
    assert np.array_equal(np.cumprod(got[:, at] != SENT, axis=0).astype(bool), live)
    assert np.array_equal(got[:, at][live], at[want[live]])
    assert (got[0, np.setdiff1d(i[::997], at)] == SENT).all()
