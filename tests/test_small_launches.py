"""Launches from one particle up, where a wavefront's lanes are few: the FP64
engine must follow the oracle's histories exactly whatever the number of live
lanes (1 to 8 live lanes share the Philox look-ahead of a wavefront eight
ways, up to 16 four ways, up to 32 two ways, more fill their own), and a
particle that is handed from launch to launch continues where it stopped."""
import pytest

from cases import write_case
from test_device import assert_same_histories, run_both

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def D():
    from ompmc_amd import device
    return device


@pytest.mark.parametrize("ncase", [1, 8, 9, 16, 17, 32, 33, 64, 65, 257])
@pytest.mark.parametrize("case", ["electron6MeV", "slab6MV"])
def test_few_particles_replay_oracle_histories(oracle, D, tmp_path, case, ncase):
    r = run_both(oracle, D, write_case(case, tmp_path, ncase=ncase, nbatch=1))
    assert_same_histories(r, f"{case} x {ncase}")
