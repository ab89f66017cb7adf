"""A context that names no number of pipelines is made about as fast as one
that names the number it gets: it does not look for more hardware queues than
there are."""
import time

import pytest

pytestmark = pytest.mark.gpu


def test_automatic_pipelines_cost_no_search():
    from ompmc_amd import device as D

    def made(pipelines):
        t = time.perf_counter()
        eng = D.Engine(1, chunk=1 << 14, pipelines=pipelines)       # small queues: their allocation takes no time
        ms = 1e3 * (time.perf_counter() - t)
        eng.close()
        return ms

    made(0)
    named = min(made(4) for _ in range(8))
    assert min(made(0) for _ in range(8)) < 2.5 * named
