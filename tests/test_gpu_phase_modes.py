"""The constant-coefficient mode form of the phase-field passes (elements inside
one phase, taken by whole waves) beside the Gauss-point form, against the
oracle: images of one phase, of layers and of boxes, with gc = 0 regions, on
tiles that end inside and past the grid."""
import numpy as np
import pytest

import oracle as O
from gpu_common import max_rel, rel_l2, require_gpu, say

pytestmark = pytest.mark.gpu

# level-0 elements (the finest level has twice as many per axis), spacings
GRIDS = {
    "37x11x9": ((18, 5, 4), (1.0, 1.0, 1.0)),    # two tiles in x and y, the last ones past the grid
    "33x15x3": ((16, 7, 1), (0.9, 1.1, 1.3)),    # two element layers
    "33x225x7": ((16, 112, 3), (1.0, 1.0, 1.0)),  # long z-chunks
}
IMAGES = ("phase", "layers", "boxes")


@pytest.fixture(scope="module")
def HA():
    return require_gpu()


def gc_image(kind, dims, rng, void):
    nx, ny, nz = dims
    lab = np.zeros((nz, ny, nx), dtype=int)
    if kind == "layers":
        lab[nz // 2:] = 1
        lab[:, ny // 2:, :] += 1
    elif kind == "boxes":
        for _ in range(6):
            a = [int(rng.integers(0, n)) for n in lab.shape]
            lab[a[0]:a[0] + 3, a[1]:a[1] + 4, a[2]:a[2] + 9] = rng.integers(1, 4)
    return np.array([100.0, 1000.0, 70.0, 0.0 if void else 25.0])[lab]


def pair(HA, grid, kind, seed, void):
    enb, h = GRIDS[grid]
    dom = tuple(v for i in range(3) for v in (0.0, 2.0 * enb[i] * h[i]))
    o, s = O.Oracle(1, enb, dom, lc=2.0), HA.Solver(1, enb, dom, lc=2.0)
    rng = np.random.default_rng(seed)
    gc = gc_image(kind, o.dims(1), rng, void)
    H = rng.uniform(0, 50, gc.shape)
    for obj in (o, s):
        obj.set(O.GC, 1, gc)
        obj.set(O.H, 1, H)
    return o, s, rng, gc.shape


# bounds: test_gpu_parity's of the same operator and smoother
@pytest.mark.parametrize("kind", IMAGES)
@pytest.mark.parametrize("grid", GRIDS)
def test_operator(HA, grid, kind):
    say(f"[gpu] phase-field modes, operator {grid} {kind}")
    o, s, rng, shape = pair(HA, grid, kind, 51, void=True)
    x = rng.standard_normal(shape)
    for obj in (o, s):
        obj.set(O.PD, 1, x)
        obj.fld(1, O.PD, O.WD)
    assert max_rel(s.get(O.WD, 1), o.field(O.WD, 1)) < 1e-12


@pytest.mark.parametrize("kind", IMAGES)
@pytest.mark.parametrize("grid", GRIDS)
def test_smoother(HA, grid, kind):
    say(f"[gpu] phase-field modes, smoother {grid} {kind}")
    o, s, rng, shape = pair(HA, grid, kind, 52, void=False)
    d0, fd = rng.uniform(0, 0.5, shape), rng.standard_normal(shape)
    for obj in (o, s):
        obj.set(O.D, 1, d0)
        obj.set(O.FD, 1, fd)
        obj.pcg_d(1, 3)
    assert rel_l2(s.get(O.D, 1), o.field(O.D, 1)) < 1e-11
    assert rel_l2(s.get(O.RD, 1), o.field(O.RD, 1)) < 1e-10
