"""Fields that overflow, in the reference's CPU form (no Debye term).

The reference replaces NaN by 0 where a field turns out NaN, so what a cell
does after an overflow is part of its behaviour: the CPU form has no
polarisation current that an infinite Ez could spoil.  The permittivities are
so small that a patch's curl coefficient overflows Ez within a few steps.

The general row sweep (grids under 64 columns) and the register tiles advance
the same disc in grids of different sizes; until the wave has been to the
nearest CPML strip and back, what lies around the disc must be the same bit for
bit, NaN and infinities included, and Jp must be zero everywhere."""
import numpy as np
import pytest

import tomography_amd as t
from cases import ref_cpu_small

STEPS, RADIUS = 24, 9.5
CROP = 14  # cells either side of the centre


def disc(n, flags):
    c = ref_cpu_small(steps=STEPS, n=n)
    return c.copy(ncpml=4, breast_radius=RADIUS * c.dx, numpatches=3, n_params=18, pulse_t0=0.0, flags=flags)


def crop(field, n):
    return field[n // 2 - CROP:n // 2 + CROP, n // 2 - CROP:n // 2 + CROP]


def test_the_crop_is_out_of_reach_of_the_strips():
    """From the disc to the strip of the smallest grid and back to the crop
    takes longer than the run (one cell a step)."""
    half = 60 // 2
    assert (half - 4 - RADIUS) + (half - 4 - CROP) > STEPS


@pytest.mark.gpu
@pytest.mark.parametrize("clamp", [True, False])
@pytest.mark.parametrize("n", [64, 67, 100])
def test_overflowing_fields_equal_the_row_sweep(n, clamp):
    flags = t.FLAG_CPU_REF_VARIANT & ~t.FLAG_FWF_ABS_ORIGIN  # the pulse by offsets from the centre
    if clamp:
        flags &= ~t.FLAG_NO_NAN_CLAMP
    rng = np.random.default_rng(8)
    p = np.concatenate([10.0 ** rng.uniform(-30, 0, 9), rng.uniform(0.0, 0.3, 9)])
    out = []
    for size in (60 + n % 2, n):  # the centre node's place depends on the parity
        cfg = disc(size, flags)
        with t.Context() as c:
            c.set_schedule(tsteps=4, chunk=4, form=t.FORM_FUSED)
            g = c.sim(cfg, p, exc=1)
            mid = []
            for _ in range(STEPS // 4):
                g.step(4)
                mid.append(g.fields())
            mat = g.materials()[0]
            g.close()
        out.append((size, mid, mat))
    (na, a, mat_a), (nb, b, mat_b) = out
    assert np.array_equal(crop(mat_a, na), crop(mat_b, nb))
    overflowed = False
    for fa, fb in zip(a, b):
        for name, x, y in zip(("ez", "hx", "hy", "jp"), fa, fb):
            assert np.array_equal(crop(x, na), crop(y, nb), equal_nan=True), name
        overflowed |= not np.all(np.isfinite(crop(fa[0], na)))
        assert not fa[3].any() and not fb[3].any()
    assert overflowed
