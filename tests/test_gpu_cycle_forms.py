"""Cycle parameters beyond one post-smoothing call and gamma 1, whose smoother
calls start from what the call or transfer before them left (cycle_d: nu2 calls
of nu2 iterations, the next cycle's first call; without post-smoothing every
call on its own; second visits of a coarse level at gamma 2), against the
oracle, and as graph replays and fused launches against kernel by kernel."""
import threading

import numpy as np
import pytest

import oracle as O
from gpu_common import make_pair, rel_l2, require_gpu, say

pytestmark = pytest.mark.gpu

# 9x9x5 nodes in one workgroup, 17x17x9 by tile passes, 33x33x17
ML, ENB, DOM = 2, (8, 8, 4), (0.0, 32.0, 0.0, 32.0, 0.0, 16.0)
NCY = 3
MG_D = [(10, 2, 3, 1), (6, 1, 2, 2), (10, 2, 0, 1), (4, 0, 1, 1)]
MG_U = [(6, 4, 2, 2), (6, 2, 0, 1), (6, 0, 3, 1), (50, 4, 2, 2)]


@pytest.fixture(scope="module")
def HA():
    return require_gpu()


def pair(HA, mg_u=(6, 4, 2, 1), mg_d=(10, 2, 1, 1), ncy=NCY):
    # tolerances that ncy cycles do not reach
    kw = dict(lc=2.0, small_k=1e-6, tol_u=1e-60, tol_d_rel=1e-60, tol_d_abs=1e-80, mg_u=mg_u + (ncy,),
              mg_d=mg_d + (ncy,))
    o, s, _ = make_pair(HA, ML, ENB, DOM, seed=80, lab_incl=4, **kw)
    return o, s


def set_phase(obj):
    """strain history, right-hand sides and d = 0"""
    dims = obj.dims(ML)
    rng = np.random.default_rng(81)
    obj.set(O.H, ML, rng.uniform(0, 20, dims[::-1]))
    obj.voigt_all_level(O.H)
    for l in range(ML, -1, -1):
        obj.fd_h(l)
    obj.set(O.D, ML, np.zeros(dims[::-1]))


def close_history(a, b, scale, tol):
    """residual norms (squared in the histories) within tol of |scale|"""
    a, b = np.sqrt(np.asarray(a)), np.sqrt(np.asarray(b))
    return len(a) == len(b) and np.max(np.abs(a - b)) <= tol * np.sqrt(scale)


@pytest.mark.parametrize("mg", MG_D, ids=str)
def test_phase_field_cycles(HA, mg):
    say(f"[gpu] phase-field cycles mg_d={mg}")
    o, s = pair(HA, mg_d=mg)
    for obj in (o, s):
        set_phase(obj)
    fo, co = o.phase_field(0, 0.0)
    fs, cs = s.phase_field(0, 0.0)
    assert co == cs == NCY
    # the bounds of test_gpu_parity's single cycle; the residual's rounding is
    # that of the first one, of which the last cycles leave little
    assert fs == pytest.approx(fo, rel=1e-12)
    ho = o.history("d")
    assert close_history(s.history(), ho, ho[0], 1e-12), (s.history(), ho)
    assert rel_l2(s.get(O.D, ML), o.field(O.D, ML)) < 1e-10


@pytest.mark.parametrize("mg", MG_U, ids=str)
def test_mechanical_cycles(HA, mg):
    say(f"[gpu] mechanical cycles mg_u={mg}")
    o, s = pair(HA, mg_u=mg)
    fo, co = o.u_entire(1.0, 0, 0.0)
    fs, cs = s.u_entire(1.0, 0, 0.0)
    assert co == cs == NCY
    # the bounds of test_gpu_parity's single cycle
    assert fs == pytest.approx(fo, rel=1e-7)
    assert close_history(s.history(), o.history("u"), fo, 1e-7), (s.history(), o.history("u"))
    assert rel_l2(s.get(O.U, ML), o.vec(O.U, ML)) < 1e-9


def solve(s):
    for c in range(3):
        s.fill(O.U, ML, 0.0, c)
        s.fill(O.FU, ML, 0.0, c)
    s.fill(O.D, ML, 0.0)
    out = [s.u_entire(1.0, 0, 0.0), s.history().tolist()]
    set_phase(s)
    out += [s.phase_field(0, 0.0), s.history().tolist()]
    return out, s.get(O.U, ML), s.get(O.D, ML)


def same(a, b):
    return a[0] == b[0] and np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])


@pytest.mark.parametrize("i", range(4))
def test_graph_replays_identical(HA, i):
    say(f"[gpu] graphs: mg_u={MG_U[i]} mg_d={MG_D[i]}")
    _, s = pair(HA, MG_U[i], MG_D[i])
    alone = solve(s)
    s.set_graphs(True)
    for _ in range(2):
        got = solve(s)
        assert same(alone, got), f"{alone[0]} {got[0]}"


@pytest.mark.parametrize("i", range(4))
def test_fused_launches_identical(HA, i):
    say(f"[gpu] fused: mg_u={MG_U[i]} mg_d={MG_D[i]}")
    fz = HA.Fuser(window_us=20000)
    two = [pair(HA, MG_U[i], MG_D[i], 10)[1] for _ in range(2)]
    alone = solve(two[0])
    got = [[], []]
    gate = threading.Barrier(2)
    for t in two:
        t.set_fuser(fz)

    def run(k):
        for _ in range(6):
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
        assert same(alone, g), f"{alone[0]} {g[0]}"
    assert len(got[0]) == len(got[1]) == 6
