"""Pinned result buffers belong to submitted requests: a context that runs
fields pins none, one request at a time pins one, a burst two.  They are
mappings of the device file of just the size of a result (sum and sum of
squares of every region)."""
import numpy as np
import pytest

from ompmc_amd import configs as cfg
from test_serving import drain

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def D():
    from ompmc_amd import device
    return device


def mappings(nbytes):
    n = 0
    with open("/proc/self/maps") as f:
        for line in f:
            lo, hi = (int(x, 16) for x in line.split()[0].split("-"))
            n += "/dev/dri" in line and nbytes <= hi - lo < nbytes + 16384
    return n


def test_result_buffers_are_pinned_for_requests_only(oracle, D, tmp_path):
    pf = cfg.water_cube(97, 24.0).write_egsphant(tmp_path / "p.egsphant")      # 14.6 MB a result: no other buffer's size
    cfg.write_inp(tmp_path / "e", cfg.dosxyz_inp_items(tmp_path, pf, ncase=10))
    pp = oracle.load_problem(tmp_path / "e")
    nreg = pp.reg.nreg
    pinned = []
    with D.Engine(1, chunk=1 << 14, pipelines=2) as eng:
        eng.upload_media(pp.tab)
        before = mappings(16 * nreg)
        pid = eng.upload_phantom(pp.ph, pp.reg)
        pinned.append(mappings(16 * nreg) - before)
        ref, ref2 = eng.run_dosxyz(pid, pp.src, 2000, 10, seed=(1, 5), nreg=nreg)[:2]
        pinned.append(mappings(16 * nreg) - before)
        for count in (1, 1, 5):
            tickets = [eng.submit(pid, pp.src, 20000, nbatch=10, seed=(1, 5)) for _ in range(count)]
            out = drain(eng, list(tickets), dict.fromkeys(tickets, nreg))
            pinned.append(mappings(16 * nreg) - before)
            for t in tickets:
                assert out[t][0].status == 0
                assert np.allclose(out[t][1], ref, rtol=1e-10, atol=1e-10 * ref.max())
                assert np.allclose(out[t][2], ref2, rtol=1e-10, atol=1e-10 * ref2.max())
    assert pinned == [0, 0, 1, 1, 2]
    oracle.free_problem(pp)
