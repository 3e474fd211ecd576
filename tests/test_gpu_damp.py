"""GPU: Graves-Qs and the sponge on one solver, in the one pass over the wavefield
that applies both, on rows wider than a block and sponge blocks that share edges,
corners and ghost points, against the oracle stepped with orc_graves_qs and then
orc_ablexp_apply after every step (drv_rk_curv_col.c:414-416, 482-486).  The sponge
alone is equal bit for bit; with Graves-Qs the exponentials differ by an ulp on a
few inputs in 10^5, so relative L2 <= 1e-6."""
import numpy as np
import pytest

from tests import cases as cs
from tests.test_ablexp_oracle import masks
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

NSTEP, DT, FREQ = 6, 0.004, 2.0
NI, NJ, NK = 71, 18, 14


def _blocks():
    nx, ny, nz = NI + 6, NJ + 6, NK + 6
    return np.array([[1, 0, 9, 0, ny - 1, 0, nz - 1], [1, nx - 8, nx - 1, 0, ny - 1, 0, nz - 1],
                     [1, 0, nx - 1, 0, 6, 0, nz - 1], [0, 0, 0, 0, 0, 0, 0],
                     [1, 3, nx - 4, 3, ny - 4, 3, 8], [1, 60, 72, 12, 18, 9, 12]], np.int32)


@pytest.mark.parametrize("pad", ["0", "1"])
@pytest.mark.parametrize("medium,qs_on,sponge_on", [("iso", 1, 1), ("aniso", 1, 1), ("vti", 1, 0),
                                                    ("iso", 0, 1), ("visco", 0, 1)])
def test_attenuation_then_sponge(medium, qs_on, sponge_on, pad, monkeypatch):
    monkeypatch.setenv("CGFDH_PAD", pad)
    case = cs.make_case(NI, NJ, NK, seed=21, pml=(0,) * 6, medium=medium)
    w0 = cs.random_wavefield(case, seed=22)
    nx, ny, nz, nc = NI + 6, NJ + 6, NK + 6, cs.ncomp(case)
    qs = np.random.default_rng(23).uniform(5.0, 200.0, (nz, ny, nx)).astype(np.float32)
    ex, ey, ez = masks(nx, ny, nz, 10)
    blocks = _blocks()
    s = cs.make_solver(case, DT, NSTEP, variant=16)
    try:
        s.set_wavefield(w0)
        if qs_on:
            s.set_graves_qs(qs, FREQ)
        if sponge_on:
            s.set_ablexp(ex, ey, ez, blocks)
        s.run(0, NSTEP)
        w_g = s.wavefield()
    finally:
        s.close()
    orc, lib = po.Oracle(case), po.load_oracle()
    w = np.array(w0, np.float32).reshape(-1)
    for it in range(NSTEP):
        w, _, _ = orc.run(DT, 1, w, None, it0=it, nt_total=NSTEP)
        w = np.ascontiguousarray(w, np.float32)
        if qs_on:
            lib.orc_graves_qs(NI, NJ, NK, nc, po.ptr(w), po.ptr(qs), FREQ, DT)
        if sponge_on:
            lib.orc_ablexp_apply(nx, ny, nz, nc, po.ptr(w), po.ptr(ex), po.ptr(ey), po.ptr(ez),
                                 po.ptr(blocks))
    assert np.isfinite(w).all() and np.abs(w).max() > 0
    assert cs.rel_l2(w_g, w) <= 1e-6
    if not qs_on:
        assert np.array_equal(w_g, w)
