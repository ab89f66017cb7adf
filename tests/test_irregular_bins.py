"""Where the shortcut for ustep iterations of length 0 must not be taken: in
an energy bin whose correction to the scattering power is negative, the skin
depth is too, and the iteration of length 0 is a multiple-scattering step
(ompmc.c:5033-5046) with draws of its own.  The electrons run through the bin
and must stay the oracle's."""
import pytest

from ompmc_amd import _native as N, configs as cfg
from test_device import assert_same_histories, run_both

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def D():
    from ompmc_amd import device
    return device


@pytest.mark.parametrize("bins", [(26,), (40,), (24, 25, 40)])
def test_multiple_scattering_steps_of_length_zero(oracle, D, tmp_path, monkeypatch, bins):
    ph = cfg.water_cube(1, 16.0)           # one voxel: none of these electrons comes near its sides in these bins,
                                           # where steps of the distance to them never reach them
    pf = ph.write_egsphant(tmp_path / "p.egsphant")
    cfg.write_inp(tmp_path / "e", cfg.dosxyz_inp_items(tmp_path, pf, ncase=500, mono=1.0, charge=-1,
                                                        field=(-2, 2, -2, 2)))
    load = oracle.load_problem

    def load_irregular(stem):
        prob = load(stem)
        for k in bins:
            prob.tab.blcce0[k], prob.tab.blcce1[k] = -1.0, 0.0
        return prob
    monkeypatch.setattr(oracle, "load_problem", load_irregular)
    assert_same_histories(run_both(oracle, D, tmp_path / "e"), f"irregular bins {bins}")
