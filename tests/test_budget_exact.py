"""The device memory a request is admitted for is what it then takes: one
that fits the budget to the byte runs, with one byte less it is refused."""
import re

import pytest

from cases import write_case
from test_serving import drain

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def D():
    from ompmc_amd import device
    return device


@pytest.mark.parametrize("nbatch", [200, 201, 224])
def test_request_that_fits_the_budget_to_the_byte(oracle, D, tmp_path, nbatch):
    pp = oracle.load_problem(write_case("patient6MV", tmp_path / "p"))
    nreg = pp.reg.nreg

    def run(budget):
        with D.Engine(0, hbm_budget=budget, chunk=1024, pipelines=2) as eng:
            eng.upload_media(pp.tab)
            pid = eng.upload_phantom(pp.ph, pp.reg)
            t = eng.submit(pid, pp.src, 5 * nbatch, nbatch=nbatch)
            status = drain(eng, [t], {t: nreg})[t][0].status
            return status, D.lib().omc_dev_last_error().decode()

    small = 32 << 20
    status, why = run(small)
    assert status == -9
    need, leaves = (int(v) for v in re.search(r"needs (\d+) bytes, budget leaves (\d+)", why).groups())
    assert run(small + need - leaves)[0] == 0
    assert run(small + need - leaves - 1)[0] == -9
    oracle.free_problem(pp)
