"""Charged particles that leave a medium into vacuum and come back into it:
the reference then goes straight to the fictitious-cross-section test and the
discrete interaction (ompmc.c:5347-5429), with the constants of the medium
entered.  Phantoms whose media differ in those constants, and gaps in media
other than the first."""
import numpy as np
import pytest

from ompmc_amd import _native as N, configs as cfg
from test_device import assert_same_histories, run_both

pytestmark = pytest.mark.gpu

WATER, COPPER, SILVER = "H2O700ICRU", "CU700ICRU", "AG700ICRU"


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


def edge_of_flight(x0, ssd, zb):
    """x where a primary that starts at (x0, 0, zb[0]) arrives at zb[2] by two
    unscattered steps, in the transport's own operations; and whether its
    distance to that x is then no shorter than to zb[2]."""
    r = np.sqrt(ssd ** 2 + x0 ** 2)
    u, w = x0 / r, ssd / r
    x, z = x0, zb[0]
    for k in (1, 2):
        d = (zb[k] - z) / w
        before, x, z = x, x + u * d, z + w * d
    return x, z == zb[2] and (x - before) / u >= d


@pytest.mark.parametrize("charge", [-1, 1])
def test_edge_of_another_medium_between_two_gaps(oracle, D, tmp_path, charge):
    """Water, vacuum, a step of length 0 in copper (whose energy bins are
    others), vacuum, water: the particle flies exactly to an edge of the
    copper, so that it enters it and leaves it again without a step in it.
    What follows a fictitious rejection starts from water's energy bin."""
    zb = np.array([0.0, 1.0, 2.0, 3.0, 4.0, 5.0])
    x0, edge, ok = 0.3, 0.0, False
    while not ok:
        x0 += 0.001
        edge, ok = edge_of_flight(x0, 100.0, zb)
    ph = cfg.water_cube(5, 5.0)
    ph.names = [COPPER, WATER]
    ph.zb = zb
    ph.xb = np.array([-3.0, -2.0, -1.0, 0.0, edge, 3.0])
    ph.yb = np.array([-3.0, -2.0, -1.0, 1.0, 2.0, 3.0])
    ph.med[:], ph.rho[:] = 2, 1.0
    ph.rho[0] = 1.0e-7                     # the first step ends at its voxel's far side, unscattered
    ph.med[1:3], ph.rho[1:3] = 0, 0.0
    ph.med[2, :, :4], ph.rho[2, :, :4] = 1, 8.96
    pf = ph.write_egsphant(tmp_path / "edge.egsphant")
    cfg.write_inp(tmp_path / "edge", cfg.dosxyz_inp_items(tmp_path, pf, ncase=2000, mono=6.0, charge=charge,
                                                          field=(x0, x0, 0.0, 0.0)))
    r = run_both(oracle, D, tmp_path / "edge")
    assert r["cnt"].n_fict > 100
    assert_same_histories(r, f"edge between gaps, charge {charge}")
