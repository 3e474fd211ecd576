"""GPU: device volumes whose rows are padded to cache lines, as large grids have
them, for what reads, writes or indexes the volumes: the borrowed tests' grids are
small, so their rows are packed otherwise."""
import numpy as np
import pytest

from tests import test_gpu_async_output as out_async
from tests import test_gpu_batch as batch
from tests import test_gpu_dd as dd
from tests import test_gpu_force as force
from tests import test_gpu_nan_check as nan
from tests import test_gpu_output as out
from tests import test_gpu_parity as par

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def padded_rows(monkeypatch):
    monkeypatch.setenv("CGFDH_PAD", "1")


@pytest.mark.parametrize("medium,variant", par.MEDIUM_VARIANTS)
def test_every_variant(medium, variant):
    par.test_onestage_all_pairs("free_pml5", True, (1, 1, 1, 1, 1, 0), medium, variant)


@pytest.mark.parametrize("medium", ["iso", "vti", "aniso", "visco"])
def test_setup(medium):
    par.test_device_setup_matches_oracle(medium)


@pytest.mark.parametrize("medium", ["iso", "visco"])
def test_outputs(medium):
    out.test_subvolume_and_strain_match_oracle(medium)
    nan.test_first_nan_in_scan_order(medium, (20, 18, 14))


def test_outputs_beside_the_run():
    out_async.test_async_output_matches_sync()


@pytest.mark.parametrize("medium", ["iso", "visco"])
def test_dd_sources(medium):
    dd.test_dd_run_matches_oracle(medium, 16)


@pytest.mark.parametrize("medium", ["iso", "vti", "aniso", "visco"])
def test_surface_forces(medium):
    force.test_strict_surface_force_run_matches_oracle(medium, 16 if medium != "aniso" else 18, True)


def test_batch():
    batch.test_batch_matches_oracle()
    batch.test_batch_autotune_leaves_the_state()


@pytest.mark.parametrize("medium", ["iso", "vti", "visco"])
def test_fused_batch(medium, monkeypatch):
    batch.test_fused_batch_equals_individual_runs(medium, monkeypatch)


def _free():
    import torch
    return torch.cuda.mem_get_info()[0]


def _iso(ni, nj, nk):
    from cgfd3d_amd import Solver
    return Solver(ni, nj, nk, 0.004, 1, free_top=False)


def test_one_staging_buffer_for_all_solvers():
    """64 MB while solvers with padded rows live, however many, and nothing after."""
    _iso(8, 8, 8).close()
    before = _free()
    sv = [_iso(64, 60, 150) for _ in range(6)]
    made = _free()
    for s in sv:
        s.set_wavefield(np.ones(9 * s.vol, np.float32))
        s.wavefield()
    assert made - _free() <= 2 ** 22
    for s in sv:
        s.close()
    assert before - _free() <= 2 ** 25      # streams keep their queues


def test_volumes_read_by_several_threads():
    """One solver's wavefield and another's, read and written at the same time."""
    from concurrent.futures import ThreadPoolExecutor
    rng = np.random.default_rng(1)
    sv = [_iso(64, 40, 50), _iso(33, 50, 40)]
    w = [rng.random(9 * s.vol, dtype=np.float32) for s in sv]
    for s, v in zip(sv, w):
        s.set_wavefield(v)

    def work(q):
        s, v = sv[q % 2], w[q % 2]
        if q >= 4:
            s.set_wavefield(v)
        return all(np.array_equal(np.asarray(s.wavefield()).reshape(-1), v) for _ in range(12))

    with ThreadPoolExecutor(6) as ex:
        assert all(ex.map(work, range(6)))
    for s in sv:
        s.close()


def _used(make):
    f = _free()
    s = make()
    return s, f - _free()


def test_padding_is_bounded():
    """70-point rows that whole lines make 96 of: 13.9 GB of volumes, 5.2 of padding.
    Solvers are padded up to a sixteenth of the card's memory in padding, and not
    where less than an eighth of the card would be left."""
    import torch
    total = torch.cuda.mem_get_info()[1]
    packed = 4 * 49 * 70 * 1006 * 1006
    extra = 4 * 49 * 26 * 1006 * 1006
    fits = total // 16 // extra
    assert 1 <= fits and (fits + 1) * (packed + extra) < total * 3 // 4
    sv = []
    for n in range(fits + 1):
        s, used = _used(lambda: _iso(64, 1000, 1000))
        sv.append(s)
        assert abs(used - packed - (extra if n < fits else 0)) < 2 ** 28, n
    for s in sv:
        s.close()
    filler = torch.empty(_free() - total // 8 - packed, dtype=torch.uint8, device="cuda:0")
    s, used = _used(lambda: _iso(64, 1000, 1000))
    s.close()
    del filler
    torch.cuda.empty_cache()
    assert abs(used - packed) < 2 ** 28
