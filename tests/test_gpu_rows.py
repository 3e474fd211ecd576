"""GPU: device volumes whose rows are padded to cache lines, as large grids have
them, for what reads, writes or indexes the volumes: the borrowed tests' grids are
small, so their rows are packed otherwise."""
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
