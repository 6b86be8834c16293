"""Spare sample rows under a memory budget: an evaluation's simulations take
them only where they cost no further pass, and all of a pass or none."""
import numpy as np
import pytest

import tomography_amd as t
from cases import PHYS_PARAMS
from test_register_tiles import least_budget, wide

CHUNK = 60


@pytest.mark.gpu
def test_rows_make_no_further_pass():
    cfg = wide(nx=200, ny=200, n_exc=2)
    V = np.tile(PHYS_PARAMS, (6, 1))
    V[:, 0] += np.arange(6)
    T = np.zeros(cfg.farfield_len(), np.float32)
    one = least_budget(cfg, PHYS_PARAMS) * cfg.n_exc  # of one vector, without the rows (to 8 KiB)
    rows = 3 * 15 * 4 * cfg.contour_len() * cfg.n_exc
    assert rows < one / 6 and rows > 16 * 8192
    epochs = -(-cfg.steps // CHUNK)

    def run(budget):
        with t.Context(hbm_budget=budget) as c:
            c.set_schedule(tsteps=4, chunk=CHUNK)
            c.profile(True)
            D = c.eval_batch(cfg, V, target=T, want_farfield=True)[1]
            st = c.stats()
        # one projection a pass; a fold of each epoch, or of the last one alone
        return D, st["k_project_mfma"]["launches"], st["k_fold"]["launches"]

    want, passes, folds = run(0)
    assert np.abs(want).max() > 0 and (passes, folds) == (1, 1)
    for budget, expect in ((6 * one, (1, epochs)),                # all six, just
                           (6 * (one + rows), (1, 1)),            # and with the rows
                           (5 * one, (2, 2)),                     # five or four a pass: two passes either way
                           (3 * one, (2, 2 * epochs)),            # three a pass; with the rows it would be two
                           (3 * (one + rows), (2, 2)),
                           (one, (6, 6 * epochs))):
        D, *got = run(budget)
        assert tuple(got) == expect, (budget / one, got, expect)
        assert np.array_equal(D, want)
