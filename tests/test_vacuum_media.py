"""Charged particles that leave a medium into vacuum and come back into it:
the reference then goes straight to the fictitious-cross-section test and the
discrete interaction (ompmc.c:5347-5429), with the constants of the medium
entered.  Phantoms whose media differ in those constants, and gaps in media
other than the first."""
import pytest

from ompmc_amd import _native as N, configs as cfg
from test_device import assert_same_histories, run_both

pytestmark = pytest.mark.gpu

SILVER = "AG700ICRU"


@pytest.fixture(scope="module")
def D():
    from ompmc_amd import device
    return device


def both_pegs(tmp_path):
    """Media with production thresholds at 10 keV and at 189 keV in one file."""
    out = tmp_path / "both.pegs4dat"
    out.write_text("".join((N.DATA / "pegs4" / f).read_text() for f in ("521icru.pegs4dat", "700icru.pegs4dat")))
    return out


@pytest.mark.parametrize("energy,charge", [(3.0, 0), (12.0, 0), (6.0, -1), (4.0, 1)])
def test_gaps_in_second_and_third_medium(oracle, D, tmp_path, energy, charge):
    """Gaps inside the second medium, inside the third and between the two;
    the first medium's Moller threshold, atomic number and screening
    coefficients are none of theirs."""
    ph = cfg.water_cube(10, 5.0)
    ph.names = ["H2O521ICRU", "LUNG700ICRU", SILVER]
    ph.med[1:5], ph.med[5:] = 2, 3
    ph.rho[:], ph.rho[1:5], ph.rho[5:] = 0.3, 0.26, 1.5
    for gap in ((slice(2, 3), slice(2, 8), slice(2, 8)), (slice(4, 6), slice(0, 10), slice(0, 5)),
                (slice(7, 8), slice(2, 8), slice(2, 8))):
        ph.med[gap], ph.rho[gap] = 0, 0.0
    pf = ph.write_egsphant(tmp_path / "gaps.egsphant")
    items = cfg.dosxyz_inp_items(tmp_path, pf, ncase=2000, mono=energy, charge=charge, field=(-1, 1, -1, 1))
    items["pegs file"] = both_pegs(tmp_path)
    cfg.write_inp(tmp_path / "gaps", items)
    r = run_both(oracle, D, tmp_path / "gaps")
    assert_same_histories(r, f"gaps, {energy} MeV charge {charge}")
