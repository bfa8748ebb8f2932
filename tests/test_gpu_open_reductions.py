"""CG smoother calls on levels whose passes leave their partial sums to the
next pass (at most 1024 tile blocks) and on the first level past that, finest
and coarse, over the positions of the update groups of four, against the
oracle."""
import numpy as np
import pytest

import oracle as O
from gpu_common import make_pair, rel_l2, require_gpu, say

pytestmark = pytest.mark.gpu

# level-0 elements: level 0 runs the tile passes too (more nodes than the
# one-workgroup smoother takes), level 1 is the finest
CASES = {
    "33x33x17": (16, 16, 8),    # 90 tile blocks
    "41x85x61": (20, 42, 30),   # 806: more partials than threads
    "65x65x73": (32, 32, 36),   # 1110: ticketed; its level 0 open
}


@pytest.fixture(scope="module")
def HA():
    return require_gpu()


@pytest.mark.parametrize("name", CASES)
def test_smoothers(HA, name):
    enb = CASES[name]
    say(f"[gpu] open reductions {name}")
    dom = tuple(v for e in enb for v in (0.0, 2.0 * e))
    o, s, _ = make_pair(HA, 1, enb, dom, seed=71, lab_incl=2, lc=2.0)
    rng = np.random.default_rng(72)
    for l, calls in ((0, (1, 2, 4, 5)), (1, (1, 3))):
        shape = o.dims(l)[::-1]
        sets = [(O.H, rng.uniform(0, 20, shape))]
        if l == 0:
            sets += [(O.KE, rng.uniform(1e3, 5e4, shape)), (O.GE, rng.uniform(1e3, 3e4, shape))]
        u0, f0 = rng.standard_normal((3,) + shape) * 0.1, rng.standard_normal((3,) + shape) * 1e3
        d0, fd = rng.uniform(0, 0.5, shape), rng.standard_normal(shape)
        for nb in calls:
            for obj in (o, s):
                for f, a in sets + [(O.U, u0), (O.FU, f0), (O.D, d0), (O.FD, fd)]:
                    obj.set(f, l, a)
            o.pcg_u(l, nb, 0.3, 1, 1.0)
            s.pcg_u(l, nb, 0.3, 1, 1.0)
            # the bounds of test_gpu_parity's smoothers
            assert rel_l2(s.get(O.U, l), o.vec(O.U, l)) < 1e-11, f"u level {l} nb={nb}"
            assert rel_l2(s.get(O.RU, l), o.vec(O.RU, l)) < 1e-10, f"r level {l} nb={nb}"
            assert s.pcg_d(l, nb) == pytest.approx(o.pcg_d(l, nb), rel=1e-12)
            assert rel_l2(s.get(O.D, l), o.field(O.D, l)) < 1e-11, f"d level {l} nb={nb}"
            assert rel_l2(s.get(O.RD, l), o.field(O.RD, l)) < 1e-10, f"R level {l} nb={nb}"
