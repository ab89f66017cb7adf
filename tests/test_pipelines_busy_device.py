"""A context that names no number of pipelines takes as many as there are
hardware queues for, also while another context keeps the device busy.  The
number shows in the device memory that the pipelines' queues leave of a
budget.  HIP reads GPU_MAX_HW_QUEUES once, so this runs in a process of its
own."""
import os
import subprocess
import sys
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu

ROOT = Path(__file__).resolve().parents[1]

SCRIPT = """
import re, sys, tempfile, threading, time
sys.path[:0] = [{root!r}, {root!r} + "/oracle", {root!r} + "/tests/golden"]
from pathlib import Path
import pyoracle as O
from ompmc_amd import device as D, _native as N
from cases import write_case
N.ensure_spinms()
pp = O.load_problem(write_case("slab6MV", Path(tempfile.mkdtemp())))

def left(pipelines, made=lambda: None):
    with D.Engine(1, hbm_budget=1 << 30, chunk=1 << 14, pipelines=pipelines, tally_bytes=-1) as eng:
        made()
        eng.upload_media(pp.tab)
        pid = eng.upload_phantom(pp.ph, pp.reg)
        eng.submit(pid, pp.src, 400000, nbatch=400000)      # cannot fit
        eng.step()
        return int(re.search(r"budget leaves (\\d+)", D.lib().omc_dev_last_error().decode()).group(1))

of = {{left(n): n for n in (4, 5, 6)}}
print("idle", of[left(0)], flush=True)
with D.Engine(1) as eng:
    eng.upload_media(pp.tab)
    pid = eng.upload_phantom(pp.ph, pp.reg)
    for k in range(8):
        run = threading.Thread(target=lambda: eng.run_dosxyz(pid, pp.src, 80000000, 10, nreg=pp.reg.nreg))
        run.start()
        time.sleep(0.02 + 0.01 * k)
        running = []
        n = of[left(0, lambda: running.append(run.is_alive()))]
        print("busy" if running[0] else "late", n, flush=True)
        run.join()
"""


def test_pipelines_of_a_context_made_beside_a_busy_one():
    r = subprocess.run([sys.executable, "-u", "-c", SCRIPT.format(root=str(ROOT))],
                       env=dict(os.environ, GPU_MAX_HW_QUEUES="16"),
                       capture_output=True, text=True, timeout=90)
    assert r.returncode == 0, r.stderr[-2000:]
    got = [line.split() for line in r.stdout.splitlines()]
    assert sum(what == "busy" for what, _ in got) > 3, r.stdout
    assert {int(n) for _, n in got} == {6}, r.stdout
