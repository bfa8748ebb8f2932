"""The mixed solve over a coarsest level of 616 nodes and 420 elements, which
takes the FP64 tile passes with the Gauss-point sums above Chebyshev degree 2
and one workgroup else: against the direct solution, and two such solves at
once through the fuser against one alone."""
import threading

import numpy as np
import pytest

import oracle as O
from gpu_common import make_pair, material_from_labels, require_gpu, say
from test_gpu_mixed import KW, direct_solution, err_modulo_rotation, rotation_mode, zero_u

pytestmark = pytest.mark.gpu

# unequal spacings, so that every scale of the element differs; the cubic
# grid folds them into the moduli
GRIDS = {"cubic": (0.0, 12.0, 0.0, 20.0, 0.0, 14.0), "box": (-1.0, 9.8, 0.0, 22.0, 0.5, 18.7)}
ML, ENB = 1, (6, 10, 7)
DEGREES = {"degree2": dict(cheb_degree=2), "degree4": dict(cheb_degree=4, cheb_ratio=12.0, cheb_upper=1.3),
           "degree4-f64": dict(cheb_degree=4, cheb_ratio=12.0, cheb_upper=1.3, precond_fp64=True)}


@pytest.fixture(scope="module")
def HA():
    return require_gpu()


@pytest.mark.parametrize("form", DEGREES)
@pytest.mark.parametrize("grid", GRIDS)
def test_matches_direct_solve(HA, grid, form):
    dom = GRIDS[grid]
    say(f"[gpu] mixed, coarsest level of 616 nodes, {grid} {form}")
    o, s, lab = make_pair(HA, ML, ENB, dom, seed=90, lab_incl=4, **KW)
    K, G, _ = material_from_labels(lab)
    dims, h = o.dims(ML), o.h(ML)
    zero = np.zeros(dims[::-1])
    ud, _, _ = direct_solution(dims, h, dom, K, G, zero, zero, 1.0, KW["small_k"])
    zero_u(s, ML)
    fs, it = s.u_entire_mixed(1.0, 0, 0.0, tol=1e-22, max_iter=200, **DEGREES[form])
    rel = s.last_stats.r_norm_final / fs
    err = err_modulo_rotation(s.get(O.U, ML), ud, rotation_mode(dims, h, dom))
    say(f"  {it} iterations, squared rel residual {rel:.3e}, rel L2 error {err:.3e}")
    # the bounds of test_gpu_mixed's direct solves
    assert rel <= 1e-22 and it < 200
    assert err < 1e-9


@pytest.mark.parametrize("form", DEGREES)
def test_fused_identical(HA, form):
    say(f"[gpu] mixed, coarsest level of 616 nodes, fused, {form}")
    two = [make_pair(HA, ML, ENB, GRIDS["cubic"], seed=91, lab_incl=4, **KW)[1] for _ in range(2)]

    def solve(s):
        zero_u(s, ML)
        return s.u_entire_mixed(1.0, 0, 0.0, tol=1e-20, max_iter=200, **DEGREES[form]), s.history().tolist(), \
            s.get(O.U, ML)

    alone = solve(two[0])
    fz = HA.Fuser(window_us=20000)
    got = [[], []]
    gate = threading.Barrier(2)
    for t in two:
        t.set_fuser(fz)

    def run(k):
        for _ in range(4):
            gate.wait(timeout=60)
            got[k].append(solve(two[k]))

    th = [threading.Thread(target=run, args=(k,)) for k in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join(timeout=100)
    assert not any(t.is_alive() for t in th), "a fused solve did not return"
    st = fz.stats()
    for t in two:
        t.close()
    fz.close()
    assert st["max_problems"] == 2, st
    for g in got[0] + got[1]:
        assert g[:2] == alone[:2] and np.array_equal(g[2], alone[2])
    assert len(got[0]) == len(got[1]) == 4
