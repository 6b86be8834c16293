"""The register-tile update against the row sweeps and the oracle.

A context under an installed streams schedule advances a simulation by itself
with the row-sweep kernels; the fused form takes register tiles.  Every cell
must come out the same bit for bit: on grids of exactly one tile (64 x 32
nodes and one more), odd and non-square ones, material, source and contour in
edge tiles, thin and thick CPML, and DFT chunks that end in a shorter block.
Reference-compatible simulations (register tiles under every form) are held to
the FP32 oracle's field tolerance."""
import numpy as np
import pytest

import tomography_amd as t
from cases import PHYS_PARAMS, fat_medium, phys_small, ref_cpu_params, ref_cpu_small, ref_params, ref_small, rel_l2

FIELD_TOL_F32 = 1e-5  # relative L2 against the FP32 oracle, as in test_gpu_parity


def tiny(nx, ny):
    c = t.preset(t.PRESET_CFG4, 64)
    return c.copy(nx=nx, ny=ny, steps=130, n_freq=2, n_angles=24, ncpml=5, ntff_offset=8, breast_radius=0.005,
                  skin_thickness=0.001, src_radius=0.006)


def wide(**over):
    c = t.preset(t.PRESET_CFG1).copy(steps=170, n_freq=2, n_angles=24, n_exc=4, breast_radius=0.025, src_radius=0.03)
    return c.copy(**over)


CASES = {
    "one tile exactly": (tiny(63, 31), PHYS_PARAMS, 0),
    "one node less (row sweeps)": (tiny(62, 31), PHYS_PARAMS, 0),
    "one node more": (tiny(64, 32), PHYS_PARAMS, 0),
    "two tiles high": (tiny(63, 64), PHYS_PARAMS, 0),
    "wide": (wide(nx=301, ny=140), PHYS_PARAMS, 1),
    "tall": (wide(nx=140, ny=301), PHYS_PARAMS, 3),
    "thin CPML": (wide(nx=256, ny=256, ncpml=1, ntff_offset=3), PHYS_PARAMS, 2),
    "thick CPML": (wide(nx=256, ny=256, ncpml=31, ntff_offset=60), PHYS_PARAMS, 2),
    "contour inside the phantom": (wide(nx=256, ny=256, ntff_offset=100), PHYS_PARAMS, 1),
    "source in material, material at the edges": (*(lambda c, p: (c.copy(steps=170), p))(*fat_medium()), 0),
    "FP64 running DFT": (phys_small(steps=170, n=200, flags=t.FLAG_DFT_FP64), PHYS_PARAMS, 1),
}


@pytest.mark.gpu
@pytest.mark.parametrize("chunk", [4, 32, 60])
@pytest.mark.parametrize("name", list(CASES))
def test_register_tiles_equal_row_sweeps(name, chunk):
    cfg, p, exc = CASES[name]
    out = []
    for form in (t.FORM_STREAMS, t.FORM_FUSED):
        with t.Context() as c:
            c.set_schedule(tsteps=4, seg_rows=16, edge_waves=2, chunk=chunk, form=form)
            g = c.sim(cfg, p, exc=exc)
            g.step(37)  # an odd split: partial blocks and chunks
            g.step(cfg.steps - 37)
            out.append([*g.fields(), *g.dft(), *g.farfield()])
            g.close()
    assert np.abs(out[0][0]).max() > 0
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.gpu
def test_default_context_and_mixed_sets_equal_row_sweeps():
    """A context with no schedule installed, and sets of several grids (one of
    them too small for a tile) advancing together, against the row sweeps."""
    mix = [tiny(63, 40), tiny(40, 63), wide(nx=150, ny=150, n_exc=2)]
    with t.Context() as c:
        c.set_schedule(tsteps=4, seg_rows=16, edge_waves=2, chunk=32, form=t.FORM_STREAMS)
        want = [c.eval(cfg, PHYS_PARAMS) for cfg in mix]
    with t.Context() as c:
        assert [c.eval(cfg, PHYS_PARAMS) for cfg in mix] == want
        for pick in ((0, 1, 2), (0, 2)):
            tickets = [c.submit(mix[i], PHYS_PARAMS) for i in pick]
            assert [c.wait(k)[0] for k in tickets] == [want[i] for i in pick]


@pytest.mark.gpu
@pytest.mark.parametrize("n, cpu", [(83, False), (132, True), (260, False)])
def test_reference_register_tiles_vs_oracle(oracle, n, cpu):
    cfg, p = (ref_cpu_small(steps=240, n=n), ref_cpu_params(4)) if cpu else (ref_small(steps=240, n=n), ref_params(5))
    with t.Context() as c:
        g = c.sim(cfg, p, exc=2)
        g.step(101)
        g.step(139)
        got = g.fields()
        g.close()
    o = oracle.sim(cfg, p, exc=2)
    o.step(240)
    for name, a, b in zip(("ez", "hx", "hy"), got, o.fields()):
        assert rel_l2(a, b) < FIELD_TOL_F32, (name, rel_l2(a, b))


def test_division_by_known_kappa_is_the_division():
    """The reference stage divides by kappa in [1, 10]; the kernel multiplies by
    its 64-bit reciprocal and rounds once, which is the 32-bit quotient itself."""
    rng = np.random.default_rng(3)
    k = np.concatenate([rng.uniform(1, 10, 4000), [1, 2, 3, 7, 9.999999]]).astype(np.float32)
    a = np.concatenate([rng.uniform(-1, 1, 4000), np.nextafter(np.float32(1), np.float32(2)) * np.ones(5)])
    for e in (-120, -60, -1, 0, 40, 120):
        x = (a * 2.0 ** e).astype(np.float32)
        with np.errstate(all="ignore"):
            assert np.array_equal((x[:, None].astype(np.float64) * (1.0 / k.astype(np.float64))).astype(np.float32),
                                  x[:, None] / k)


def least_budget(cfg, p):
    """Smallest memory budget (to 4 KiB) under which the simulation is accepted."""
    lo, hi = 0, t.request_bytes(cfg) * 2 // 4096
    while hi - lo > 1:
        mid = (lo + hi) // 2
        try:
            with t.Context(hbm_budget=mid * 4096) as c:
                c.set_schedule(tsteps=4, chunk=60)
                c.sim(cfg, p).close()
            hi = mid
        except t.TomoError:
            lo = mid
    return hi * 4096


@pytest.mark.gpu
@pytest.mark.parametrize("chunk", [4, 32, 64])
@pytest.mark.parametrize("name", ["one tile exactly", "wide", "thick CPML", "FP64 running DFT"])
def test_fold_in_the_next_epoch_equals_its_own_launch(name, chunk):
    """Evaluations fold an epoch's samples in the next epoch's first launch,
    stepped simulations in a launch of their own: the same far field, for
    chunks shorter than the longest block, runs that end in a partial chunk and
    several simulations together."""
    cfg, p, exc = CASES[name]
    cfg = cfg.copy(steps=cfg.steps + 3 * chunk)
    T = np.zeros(cfg.farfield_len(), np.float32)
    with t.Context() as c:
        c.set_schedule(tsteps=4, chunk=chunk, form=t.FORM_FUSED)
        want = []
        for e in range(cfg.n_exc):
            g = c.sim(cfg, p, exc=e)
            g.step(cfg.steps)
            want.append(g.farfield()[0].ravel())
            g.close()
        want = np.concatenate(want)
        for many in (1, 3):
            D = c.eval_batch(cfg, np.tile(p, (many, 1)), target=T, want_farfield=True)[1]
            assert np.abs(want).max() > 0
            for d in D:
                assert np.array_equal(d.ravel(), want)


@pytest.mark.gpu
def test_a_budget_without_room_for_spare_sample_rows():
    """A budget that just holds the simulation is still enough, and its result
    is the same."""
    cfg = wide(nx=200, ny=200, n_exc=1)
    T = np.zeros(cfg.farfield_len(), np.float32)
    got = []
    for budget in (0, least_budget(cfg, PHYS_PARAMS)):
        with t.Context(hbm_budget=budget) as c:
            c.set_schedule(tsteps=4, chunk=60)
            got.append(c.eval_batch(cfg, PHYS_PARAMS, target=T, want_farfield=True)[1])
    assert np.abs(got[0]).max() > 0
    assert np.array_equal(*got)


@pytest.mark.gpu
@pytest.mark.parametrize("n, many", [(830, 1), (1030, 1), (401, 8), (140, 40), (259, 24)])
def test_tile_order_changes_no_result(n, many):
    """Sets of more tiles than compute units are dealt by work: one grid in pairs
    of tiles, many in several rounds, 8 and 16 waves; against the row sweeps."""
    # (the contour 20 cells outside the source, so that 70 steps reach it)
    cfg = wide(nx=n, ny=n, n_exc=1, steps=70, ntff_offset=max(n // 2 - 80, 15))
    V = np.tile(PHYS_PARAMS, (many, 1))
    V[:, 0] += np.linspace(-1, 1, many)
    T = np.zeros(cfg.farfield_len(), np.float32)
    with t.Context() as c:
        c.set_schedule(tsteps=4, chunk=60, form=t.FORM_FUSED)
        D = c.eval_batch(cfg, V, target=T, want_farfield=True)[1]
    with t.Context() as c:
        c.set_schedule(tsteps=4, seg_rows=16, edge_waves=2, chunk=60, form=t.FORM_STREAMS)
        for i in sorted({0, many // 2, many - 1}):
            g = c.sim(cfg, V[i])
            g.step(cfg.steps)
            want = g.farfield()[0]
            g.close()
            assert np.abs(want).max() > 0
            assert np.array_equal(D[i].ravel(), want.ravel())
