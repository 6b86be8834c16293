"""The fused row sweep at sizes with tiles of every class.  Grids that register
tiles hold reach it when they advance in one set with a grid too small for
them; each simulation's result is the one it has by itself, on register tiles."""
import numpy as np
import pytest

import tomography_amd as t
from cases import PHYS_PARAMS
from test_register_tiles import tiny, wide
from tomography_amd.workloads import PLAIN_SCHEDULE, cell_steps


@pytest.mark.gpu
@pytest.mark.parametrize("over", [{}, dict(tsteps=2, seg_rows=12, inner_rows=0, inner_waves=4, edge_rows=5, edge_waves=2)])
def test_mixed_sets_on_the_fused_row_sweep(over):
    sched = {**PLAIN_SCHEDULE, **over}
    mix = [wide(nx=256, ny=256, n_exc=1), tiny(40, 63).copy(steps=170), wide(nx=301, ny=220, n_exc=2)]
    vec = [PHYS_PARAMS + np.array([i, 0, 0, 0, 0, 0, 0, 0]) for i in range(3)]
    with t.Context() as c:
        c.set_schedule(**sched)
        want = [c.eval(cfg, v) for cfg, v in zip(mix, vec)]
        assert all(np.isfinite(want)) and min(want) < 0
        c.profile(True)
        tickets = [c.submit(cfg, v) for cfg, v in zip(mix, vec)]
        assert [c.wait(k)[0] for k in tickets] == want
        st = c.stats()
        ran = {k: v["launches"] for k, v in st.items() if k.startswith("k_t") and v["launches"]}
        # blocks of tsteps steps, where register tiles take ten or more
        assert ran == {"k_tfused": sum(-(-n // sched["tsteps"]) for n in (60, 60, 50))}
        assert st["update"]["cell_steps"] == sum(map(cell_steps, mix))
