"""The mixed-precision solve at every order of its iterate's updates: the
Chebyshev steps add their directions to the iterate singly or in pairs by
degree and position, in the solve's own order, so that each degree (odd and
even, 1 without a first step) must reach the converged solution."""
import numpy as np
import pytest

import oracle as O
from gpu_common import make_pair, require_gpu, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def HA():
    return require_gpu()


@pytest.mark.parametrize("form", [dict(), dict(precond_fp64=True), dict(element_mfma=True)],
                         ids=["f32", "f64", "f32-mfma"])
def test_degrees(HA, form):
    ml, enb, dom = 2, (4, 4, 4), (0.0, 16.0, 0.0, 16.0, 0.0, 16.0)
    _, s, _ = make_pair(HA, ml, enb, dom, seed=61, lab_incl=4, lc=2.0, tol_u=1e-16, mg_u=(50, 4, 2, 1, 30))
    H = []
    iters = []
    for deg in (4, 1, 2, 3, 5, 6):
        say(f"[gpu] Chebyshev degree {deg} {form}")
        for i in range(3):
            s.fill(O.U, ml, 0.0, i)
            s.fill(O.FU, ml, 0.0, i)
        fs, it = s.u_entire_mixed(1.0, 0, 0.0, tol=1e-22, max_iter=200, cheb_degree=deg, cheb_ratio=6.0, **form)
        assert s.last_stats.r_norm_final / fs <= 1e-22 and it < 200
        # the strain energy's limit is free of the rotation the boundary leaves
        H.append(np.array([s.U_e(), s.externe_force_sum()]))
        iters.append(it)
    say(f"  outer iterations by degree 4, 1, 2, 3, 5, 6: {iters}")
    # relative residual 1e-11 at a condition that test_gpu_mixed's solutions
    # keep below 1e-9 of the direct one
    for h in H[1:]:
        assert np.all(np.abs(h - H[0]) <= 1e-9 * np.abs(H[0]))
    # a step that lost or doubled a direction would not precondition: the outer
    # iterations fall as the degree rises
    assert iters[0] <= iters[2] <= iters[1] and iters[5] <= iters[3]
