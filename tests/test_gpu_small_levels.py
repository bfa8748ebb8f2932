"""The one-workgroup smoother of small levels (small_pcg_kernel) against the
oracle, at the edges of its thread layouts: the most nodes and elements of
each layout, one past them, and the first level that runs the tile passes."""
import numpy as np
import pytest

import oracle as O
from gpu_common import make_pair, rel_l2, require_gpu, say

pytestmark = pytest.mark.gpu

# level-0 elements (level 1, the finest, has twice as many per axis)
CASES = {
    "128-nodes": (7, 3, 3),      # 128 / 63: one component per thread, 3 x 128 threads
    "144-nodes": (2, 2, 15),     # 144 / 60: 3 x 256 threads
    "256-nodes": (7, 7, 3),      # 256 / 147
    "270-nodes": (2, 5, 14),     # 270 / 140: 512 threads, two nodes each
    "512-elements": (8, 8, 8),   # 729 / 512
    "513-elements": (19, 27, 1), # 1120 / 513: 1024 threads
    "1024-elements": (16, 8, 8), # 1377 / 1024
    "1530-nodes": (16, 44, 1),   # 1530 / 704
    "tile-passes": (5, 15, 14),  # 1440 / 1050: past the workgroup
}


@pytest.fixture(scope="module")
def HA():
    return require_gpu()


@pytest.mark.parametrize("name", CASES)
def test_layout_edges(HA, name):
    enb = CASES[name]
    say(f"[gpu] small level {name} {enb}")
    # anisotropic spacing, so that every scale of the element differs
    dom = (-1.0, -1.0 + 0.9 * enb[0], 0.0, 1.1 * enb[1], 0.5, 0.5 + 1.3 * enb[2])
    o, s, _ = make_pair(HA, 1, enb, dom, seed=30, lab_incl=0, lc=2.0)
    rng = np.random.default_rng(31)
    dims = o.dims(0)
    Ke = rng.uniform(1e3, 5e4, dims[::-1])
    Ge = rng.uniform(1e3, 3e4, dims[::-1])
    u0 = rng.standard_normal((3,) + dims[::-1]) * 0.1
    f0 = rng.standard_normal((3,) + dims[::-1]) * 1e3
    Hn = rng.uniform(0, 20, dims[::-1])
    d0 = rng.uniform(0, 0.5, dims[::-1])
    fd = rng.standard_normal(dims[::-1])
    # the bounds of test_gpu_parity's small levels: 4 iterations of rounding
    for nb in (0, 4):
        for obj in (o, s):
            for f, a in ((O.KE, Ke), (O.GE, Ge), (O.U, u0), (O.FU, f0), (O.H, Hn), (O.D, d0), (O.FD, fd)):
                obj.set(f, 0, a)
        o.pcg_u(0, nb, 0.3, 0, 0.0)
        s.pcg_u(0, nb, 0.3, 0, 0.0)
        assert rel_l2(s.get(O.U, 0), o.vec(O.U, 0)) < 1e-11, f"u nb={nb}"
        assert rel_l2(s.get(O.RU, 0), o.vec(O.RU, 0)) < 1e-10, f"r nb={nb}"
        fo = o.pcg_d(0, nb)
        fs = s.pcg_d(0, nb)
        assert fs == pytest.approx(fo, rel=1e-13)
        assert rel_l2(s.get(O.D, 0), o.field(O.D, 0)) < 1e-11, f"d nb={nb}"
        assert rel_l2(s.get(O.RD, 0), o.field(O.RD, 0)) < 1e-10, f"R nb={nb}"
