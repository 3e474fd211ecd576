"""GPU: the tile kernel (variant 16) where its tiles end: rows of one point past
a tile of 64 and one short of it, 8-row tiles with 1 and 7 rows left, faces whose
PML regions overlap, an aligned row that fills its lines, every medium and two to
four Maxwell bodies, from a random state with every memory variable set, against
the oracle; the same FP32 operations, so equal bit for bit."""
import numpy as np
import pytest

from oracle import pyoracle as po
from tests import cases as cs

pytestmark = pytest.mark.gpu

SHAPES = [(8, 9, 12), (63, 8, 10), (64, 15, 9), (65, 17, 11), (90, 16, 13), (130, 23, 8)]
MEDIA = ["iso", "vti", "aniso", "visco2", "visco3", "visco4"]


def _case(medium, ni, nj, nk, free, layers):
    pml = (1, 1, 1, 1, 1, 0 if free else 1)
    kind = "visco" if medium.startswith("visco") else medium
    case = cs.make_case(ni, nj, nk, seed=11, free_top=free, pml=pml, layers=layers, medium=kind)
    if kind == "visco" and medium != "visco3":
        case["med"], case["visco_wl"] = cs.visco_medium(ni, nj, nk, seed=11,
                                                        nmaxwell=int(medium[-1]))
    return case


@pytest.mark.parametrize("medium", MEDIA)
@pytest.mark.parametrize("ni,nj,nk", SHAPES)
def test_tile_edges_match_oracle(ni, nj, nk, medium):
    nt, dt = 9, 0.004
    free = (ni + nk) % 2 == 0
    case = _case(medium, ni, nj, nk, free, 5 if ni < 60 else 3)
    w, aux = cs.random_wavefield(case, seed=3).reshape(-1), cs.random_aux(case, seed=3)
    orc = po.Oracle(case)
    w_o, a_o, _ = orc.run(dt, nt, w=w, aux=aux)
    s = cs.make_solver(case, dt, nt, variant=16)
    s.set_wavefield(w)
    s.set_pml_aux(aux)
    s.run(0, nt)
    w_g, a_g = s.wavefield(), s.pml_aux()
    s.close()
    assert np.isfinite(w_o).all() and np.abs(w_o).max() > 0
    assert np.array_equal(w_g, np.asarray(w_o).reshape(-1))
    assert np.array_equal(a_g, np.asarray(a_o).reshape(-1))


@pytest.mark.parametrize("medium", MEDIA)
@pytest.mark.parametrize("ni,nj,nk", SHAPES[1::2])
def test_two_phase_steps_match_oracle(ni, nj, nk, medium, monkeypatch):
    """Variant 16 on the kernel that steps volumes past the tile kernel's reach."""
    monkeypatch.setenv("CGFDH_TILE", "0")
    test_tile_edges_match_oracle(ni, nj, nk, medium)


@pytest.mark.parametrize("medium,nk,variant", [("iso", 500, 16), ("iso", 520, 16),
                                               ("aniso", 490, 16), ("aniso", 520, 18)])
def test_default_past_the_tile_kernel(medium, nk, variant):
    """1024 x 1024 rows and planes of 506, 526 and 496: 531, 552 and 520 M points,
    either side of two volumes and a plane of 2^32 bytes (537 M)."""
    from cgfd3d_amd import MEDIUM_ELASTIC_ANISO, MEDIUM_ELASTIC_ISO, Solver
    s = Solver(1018, 1018, nk, 0.004, 1, medium_type=MEDIUM_ELASTIC_ANISO if medium == "aniso"
               else MEDIUM_ELASTIC_ISO)
    assert s.kernel_choice()[0] == variant
    s.close()
