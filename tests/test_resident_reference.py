"""Reference-compatible simulations under the resident form (the drop-in's
schedule): grids too small for register tiles advance in one cooperative
launch per DFT chunk, as fast as the form's name promises and with the row
sweep's bits; from 64 columns on the register tiles take them."""
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
