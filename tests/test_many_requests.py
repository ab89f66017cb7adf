"""Many requests admitted at once: jobs are set up from a ring of 64 pinned
stages, and the results of the first two to finish wait in pinned buffers, of
the others in ordinary memory.  Each result must be the one its request has
alone."""
import numpy as np
import pytest

from cases import write_case
from test_serving import drain

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def D():
    from ompmc_amd import device
    return device


@pytest.mark.parametrize("n", [1, 2, 3, 63, 64, 65, 130])
def test_each_of_many_requests_as_alone(oracle, D, tmp_path, n):
    pp = oracle.load_problem(write_case("slab6MV", tmp_path / "p"))
    nreg = pp.reg.nreg
    with D.Engine(1) as eng:
        eng.upload_media(pp.tab)
        pid = eng.upload_phantom(pp.ph, pp.reg)

        def submit(k):
            return eng.submit(pid, pp.src, 200 + k, nbatch=1 + k % 3, seed=(k, 5))
        tickets = [submit(k) for k in range(n)]
        got = drain(eng, list(tickets), dict.fromkeys(tickets, nreg))
        for k in {0, 1, 2, 62, 63, 64, 128, n - 1} & set(range(n)):
            t = submit(k)
            ref = drain(eng, [t], {t: nreg})[t]
            r = got[tickets[k]]
            assert r[0].status == ref[0].status == 0
            for a, b in ((r[1], ref[1]), (r[2], ref[2])):
                # sums of less than 1e5 terms in another order
                assert b.max() > 0 and np.allclose(a, b, rtol=1e-10, atol=1e-10 * b.max())
    oracle.free_problem(pp)
