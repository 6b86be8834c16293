"""Reference-compatible simulations under the resident form (the drop-in's
schedule): grids too small for register tiles advance in one cooperative
launch per DFT chunk, as fast as the form's name promises and with the row
sweep's bits; from 64 columns on the register tiles take them."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest

import tomography_amd as t
from cases import ref_params, ref_small
from tomography_amd.workloads import REF_SCHEDULE


def small(n, steps=150):
    return ref_small(steps=steps, n=n).copy(ntff_offset=3, ncpml=min(10, (n - 6) // 3), n_exc=2,
                                            breast_radius=(int(0.3 * n) + 0.5) * 1e-3)


@pytest.mark.gpu
@pytest.mark.parametrize("n, resident", [(17, True), (41, True), (62, True), (63, False)])
@pytest.mark.parametrize("tsteps, rows", [(8, 12), (4, 8)])
def test_small_reference_grids_run_resident(n, resident, tsteps, rows):
    cfg = small(n)
    T = np.zeros(cfg.farfield_len(), np.float32)
    V = np.stack([ref_params(k) for k in (1, 2, 3)])
    out = []
    for form in (t.FORM_RESIDENT, t.FORM_FUSED):
        with t.Context() as c:
            c.set_schedule(**{**REF_SCHEDULE, "tsteps": tsteps, "seg_rows": rows, "form": form})
            c.profile(True)
            D = c.eval_batch(cfg, V, target=T, want_farfield=True)[1]
            one = c.eval(cfg, V[1], target=T, want_farfield=True)[1]
            launches = c.stats()["k_tres"]["launches"]
            assert (launches > 0) == (resident and form == t.FORM_RESIDENT)
            g = c.sim(cfg, V[2], exc=1)
            g.step(37)  # a partial chunk and a partial block
            g.step(cfg.steps - 37)
            out.append([D, one, *g.fields(), *g.dft()])
            g.close()
    assert np.abs(out[0][0]).max() > 0
    assert np.array_equal(out[0][0][1], out[0][1])
    for a, b in zip(*out):
        assert np.array_equal(a, b)


_CHILD = """
import json, sys
sys.path[:0] = [{tests!r}, {root!r}]
from test_resident_reference import evaluate
f, st = evaluate()
print(json.dumps(dict(fitness=f.hex(), refused=st["resident_refused"], tres=st["k_tres"]["launches"],
                      sweep=st["k_tblock"]["launches"])))
"""


def evaluate():
    cfg = small(41)
    with t.Context() as c:
        c.set_schedule(**REF_SCHEDULE)
        c.profile(True)
        return c.eval(cfg, ref_params(4), target=np.full(cfg.farfield_len(), 0.01, np.float32)), c.stats()


@pytest.mark.gpu
def test_a_refused_process_runs_the_row_sweep():
    """A second process, which the device may refuse its cooperative queue,
    returns the same double whichever kernel it ran."""
    want, st = evaluate()
    assert st["k_tres"]["launches"] > 0 and st["resident_refused"] == 0
    tests = os.path.dirname(os.path.abspath(__file__))
    code = _CHILD.format(tests=tests, root=os.path.dirname(tests))
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    got = json.loads(r.stdout.strip().splitlines()[-1])
    assert float.fromhex(got["fitness"]) == want
    assert (got["tres"] == 0 and got["sweep"] > 0) if got["refused"] else got["tres"] > 0
