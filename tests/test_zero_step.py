"""The shortcut for ustep iterations of length 0 (transport.h, zero_ustep)
holds in the leading table bins the upload finds regular; in the others the
general iteration runs.  A positron coefficient made negative in one bin ends
the regular bins there, and electron histories, which never read it, must
stay the oracle's."""
import pytest

from ompmc_amd import _native as N, configs as cfg
from test_device import assert_same_histories, run_both

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def D():
    from ompmc_amd import device
    return device


@pytest.mark.parametrize("first_irregular", [0, 1, 150])
def test_electrons_replay_without_the_shortcut(oracle, D, tmp_path, monkeypatch, first_irregular):
    pf = cfg.slab_phantom(16, 16.0).write_egsphant(tmp_path / "p.egsphant")
    cfg.write_inp(tmp_path / "e", cfg.dosxyz_inp_items(tmp_path, pf, ncase=500, mono=1.0, charge=-1,
                                                        field=(-2, 2, -2, 2)))
    load = oracle.load_problem

    def load_irregular(stem):
        prob = load(stem)
        for m in range(prob.tab.nmed):
            prob.tab.etap_ms0[m * N.MXEKE + first_irregular] = -1.0
            prob.tab.etap_ms1[m * N.MXEKE + first_irregular] = 0.0
        return prob
    monkeypatch.setattr(oracle, "load_problem", load_irregular)
    assert_same_histories(run_both(oracle, D, tmp_path / "e"), f"irregular from bin {first_irregular}")
