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


@pytest.fixture(autouse=True)
def tiles_at_every_size(monkeypatch):
    """Small grids step on the two-phase kernel otherwise."""
    monkeypatch.setenv("CGFDH_TILE", "1")


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
    free = (ni + nk) % 2 == 0
    _match(_case(medium, ni, nj, nk, free, 5 if ni < 60 else 3), 9)


def _match(case, nt):
    dt = 0.004
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


# volumes just past the last-level cache, 256 MB, on which the kernel's accesses
# that no other point repeats are non-temporal, in 5 to 10 units of planes, the last
# one short
@pytest.mark.parametrize("medium,ni,nj,nk", [
    ("iso", 122, 100, 98), ("vti", 122, 100, 93), ("aniso", 122, 100, 71), ("visco2", 90, 90, 71),
    ("visco3", 90, 90, 55), ("visco4", 90, 90, 45)])
def test_large_volumes_match_oracle(medium, ni, nj, nk):
    case = _case(medium, ni, nj, nk, True, 7)
    nw = cs.ncomp(case)
    ncoef = 10 + len(case["med"])
    assert 4 * (4 * nw + ncoef) * (-(-(ni + 6) // 32) * 32) * (nj + 6) * (nk + 6) > 2 ** 28
    planes = nk - 4
    chunk = -(-planes // (planes // 8))
    assert planes // 8 >= 5 and planes % chunk != 0
    _match(case, 2)


@pytest.mark.parametrize("medium", MEDIA)
@pytest.mark.parametrize("ni,nj,nk", SHAPES[1::2])
def test_two_phase_steps_match_oracle(ni, nj, nk, medium, monkeypatch):
    """Variant 16 on the kernel that steps volumes past the tile kernel's reach."""
    monkeypatch.setenv("CGFDH_TILE", "0")
    test_tile_edges_match_oracle(ni, nj, nk, medium)


@pytest.mark.parametrize("pad", ["0", "1"])
@pytest.mark.parametrize("tile", ["0", "1"])
@pytest.mark.parametrize("medium", MEDIA)
def test_packed_and_padded_rows_match_oracle(medium, tile, pad, monkeypatch):
    monkeypatch.setenv("CGFDH_TILE", tile)
    monkeypatch.setenv("CGFDH_PAD", pad)
    for shape in SHAPES[2::3]:
        test_tile_edges_match_oracle(*shape, medium)


@pytest.mark.parametrize("gauss", [False, True])
@pytest.mark.parametrize("medium", ["iso", "vti", "aniso", "visco"])
def test_tile_run_with_sources_matches_oracle(medium, gauss):
    from tests.test_gpu_parity import test_run_matches_oracle
    test_run_matches_oracle(medium, 16, gauss)


@pytest.mark.parametrize("medium", ["iso", "visco"])
def test_tile_run_with_dd_sources_matches_oracle(medium):
    from tests.test_gpu_dd import test_dd_run_matches_oracle
    test_dd_run_matches_oracle(medium, 16)


def test_tile_steps_in_a_captured_batch():
    from tests import test_gpu_batch as tb
    tb.test_batch_matches_oracle()
    tb.test_batch_equals_individual_runs()


# which kernel variant 16 steps on, as the anisotropic medium's default shows it
# (18 instead of the two-phase kernel): blocks of 64 x 8 points either side of
# 1344, one round of 480 and 352 of them and two of 494, one tile between two x faces and two tiles between two y faces, rows of
# tiles that are mostly empty, 1024 x 1024 rows and planes of 506, 526 and 496
# (531, 552 and 520 M points) either side of two volumes and a plane of 2^32 bytes
# (537 M)
@pytest.mark.parametrize("medium,ni,nj,nk,x,y,variant", [
    ("aniso", 64, 64, 100, 0, 0, 18), ("aniso", 122, 122, 19, 0, 0, 16),
    ("aniso", 122, 122, 15, 0, 0, 18), ("aniso", 100, 100, 23, 0, 0, 18), ("aniso", 100, 100, 55, 0, 0, 18),
    ("aniso", 100, 100, 56, 0, 0, 16), ("aniso", 58, 200, 200, 10, 0, 18),
    ("aniso", 58, 200, 200, 15, 0, 16), ("aniso", 65, 200, 200, 10, 0, 16),
    ("aniso", 58, 200, 200, 0, 10, 16), ("aniso", 300, 16, 300, 0, 6, 18),
    ("aniso", 300, 16, 300, 6, 0, 16), ("aniso", 300, 18, 300, 0, 6, 16),
    ("aniso", 300, 11, 300, 0, 0, 18), ("aniso", 300, 12, 300, 0, 0, 16),
    ("aniso", 1018, 1018, 490, 0, 0, 16), ("aniso", 1018, 1018, 520, 0, 0, 18),
    ("iso", 1018, 1018, 500, 0, 0, 16), ("iso", 1018, 1018, 520, 0, 0, 16)])
def test_default_by_size(medium, ni, nj, nk, x, y, variant, monkeypatch):
    from cgfd3d_amd import MEDIUM_ELASTIC_ANISO, MEDIUM_ELASTIC_ISO, Solver
    monkeypatch.delenv("CGFDH_TILE")
    layers = (x, x, y, y, 0, 0)
    s = Solver(ni, nj, nk, 0.004, 1, pml_on=[n > 0 for n in layers], pml_layers=layers,
               medium_type=MEDIUM_ELASTIC_ANISO if medium == "aniso" else MEDIUM_ELASTIC_ISO)
    assert s.kernel_choice()[0] == variant
    s.close()


# 16-point rows, which whole lines would double, volumes of one Maxwell body that fit
# the last-level cache without padding only (212 and 256 MB) and of two that nearly
# do (261 and 298): packed; rows of a line's length or nearly, and large grids: on
# whole lines
@pytest.mark.parametrize("ni,nj,nk,nmaxwell,padded", [
    (10, 300, 300, 0, False), (100, 100, 60, 1, False), (50, 90, 120, 2, False),
    (209, 49, 100, 0, True), (100, 100, 60, 0, False),
    (122, 122, 60, 0, True), (100, 150, 150, 0, True)])
def test_device_memory_of_a_solver(ni, nj, nk, nmaxwell, padded, monkeypatch):
    import torch
    from cgfd3d_amd import MEDIUM_ELASTIC_ISO, MEDIUM_VISCO_ISO, Solver
    monkeypatch.delenv("CGFDH_TILE")
    Solver(8, 8, 8, 0.004, 1).close()          # code objects, static buffers
    free = torch.cuda.mem_get_info()[0]
    s = Solver(ni, nj, nk, 0.004, 1, free_top=False, nmaxwell=nmaxwell,
               medium_type=MEDIUM_VISCO_ISO if nmaxwell else MEDIUM_ELASTIC_ISO)
    used = free - torch.cuda.mem_get_info()[0]
    s.close()
    px = -(-(ni + 6) // 32) * 32 if padded else ni + 6
    vols = 4 * (9 + 6 * nmaxwell) + 10 + 3 + 2 * nmaxwell
    want = 4 * px * (nj + 6) * (vols * (nk + 6) + 36)
    # allocations are rounded to 2 MB, streams have queues, padded rows a 64 MB buffer
    assert want <= used <= want + 2 ** 25 + (2 ** 26 if px != ni + 6 else 0)
