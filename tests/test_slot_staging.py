"""Tables into a simulation and fields out of it through the pinned staging
memory, at the sizes where they take more than one piece."""
import numpy as np
import pytest

import tomography_amd as t
from cases import PHYS_PARAMS, phys_small, rel_l2

FIELD_TOL_F32 = 1e-5  # relative L2 against the FP32 oracle, as in test_gpu_parity


@pytest.mark.gpu
@pytest.mark.parametrize("nx, ny", [(511, 511), (1023, 260), (640, 700)])
def test_fields_over_row_bands(oracle, nx, ny):
    """4 MiB hold 512 rows of 512 nodes of the four fields: exactly one band, a
    last band of few rows, and several; each field alone equals the four."""
    cfg = phys_small(steps=150, n=200).copy(nx=nx, ny=ny)
    with t.Context() as c:
        g = c.sim(cfg, PHYS_PARAMS, exc=1)
        g.step(150)
        got = g.fields()
        for k, want in enumerate(got):
            one = np.full_like(want, np.nan)
            ptr = [None] * 4
            ptr[k] = one.ctypes.data_as(t.api._fp)
            assert t.api.lib().tomo_sim_fields(g.h, *ptr) == t.TOMO_OK
            assert np.array_equal(one, want)
        g.close()
    o = oracle.sim(cfg, PHYS_PARAMS, exc=1)
    o.step(150)
    for name, a, b in zip(("ez", "hx", "hy", "jp"), got, o.fields()):
        assert rel_l2(a, b) < FIELD_TOL_F32, (name, rel_l2(a, b))


@pytest.mark.gpu
def test_tables_larger_than_the_staging():
    """A waveform of 1.2 million steps (4.8 MB) is uploaded in two pieces; the
    first steps do not depend on its length."""
    short = phys_small(steps=64, n=200)
    out = []
    with t.Context() as c:
        for cfg in (short, short.copy(steps=1_200_000)):
            g = c.sim(cfg, PHYS_PARAMS, exc=1)
            g.step(64)
            out.append([*g.fields(), g.materials()[0]])
            g.close()
    assert np.abs(out[0][0]).max() > 0
    for a, b in zip(*out):
        assert np.array_equal(a, b)
