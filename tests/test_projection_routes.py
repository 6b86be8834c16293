"""The two projection kernels: few simulations take the vector-unit chains,
many (by workgroups) the matrix cores, and the far fields are the same bit for
bit; one simulation is also held to the oracle's far field by
test_gpu_parity.  Sizes: a contour leg of odd length (a pair of points on two
legs), fewer points than one tile, angles around the 8 of a workgroup, one
simulation more than a workgroup's 8, both DFT precisions."""
import numpy as np
import pytest

import tomography_amd as t
from cases import PHYS_PARAMS
from tomography_amd.workloads import seeded_vectors


def small(nx, ny, off, A, F, flags=0):
    c = t.preset(t.PRESET_CFG4, 64)
    return c.copy(nx=nx, ny=ny, steps=90, n_freq=F, n_angles=A, ncpml=5, ntff_offset=off, breast_radius=0.005,
                  skin_thickness=0.001, src_radius=0.006, n_exc=1, flags=flags)


def on_matrix_cores(n, A, F):
    return -(-A // 8) * F * -(-n // 8) >= 5000 * -(-(-(-A // 128) * F * -(-n // 32)) // 256)


@pytest.mark.gpu
@pytest.mark.parametrize("nx, ny, off, A, F, flags", [
    (70, 70, 8, 720, 8, 0), (71, 66, 9, 723, 8, 0), (64, 64, 27, 1921, 3, 0), (75, 70, 8, 720, 8, t.FLAG_DFT_FP64)])
def test_both_projections_agree(nx, ny, off, A, F, flags):
    cfg = small(nx, ny, off, A, F, flags)
    n = 65
    assert on_matrix_cores(n, A, F) and not on_matrix_cores(9, A, F)
    V = seeded_vectors(n, 8, 5)
    V[:, :3] = PHYS_PARAMS[:3]
    with t.Context() as c:
        T = np.zeros(cfg.farfield_len(), np.float32)
        many = c.eval_batch(cfg, V, target=T, want_farfield=True)[1].reshape(n, -1)
        few = c.eval_batch(cfg, V[:9], target=T, want_farfield=True)[1].reshape(9, -1)
        one = c.eval_batch(cfg, V[64:], target=T, want_farfield=True)[1].reshape(1, -1)
    assert np.abs(many).max() > 0 and np.all(np.isfinite(many))
    assert np.array_equal(many[:9], few)
    assert np.array_equal(many[64:], one)
