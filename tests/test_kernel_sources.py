"""The rule that picks a far-field projection and the reference stage's division
by a known kappa, compiled for the host from the kernel sources, so that the
tests that rest on them cannot drift from them."""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest

import test_projection_routes as routes
import tomography_amd as t
from cases import PHYS_PARAMS
from tomography_amd.workloads import seeded_vectors

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tomography_amd", "csrc")


def host_build(tmp_path, name, code):
    src = tmp_path / (name + ".cpp")
    src.write_text(code)
    lib = tmp_path / (name + ".so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-shared", "-fPIC", str(src), "-o", str(lib)], check=True)
    return ctypes.CDLL(str(lib))


def project_route(tmp_path):
    """launch_project's own rule, compiled for the host: 0 the vector units, 1 the
    matrix cores split, 2 the matrix cores."""
    text = open(os.path.join(CSRC, "kernels.hip")).read()
    const = "".join(re.findall(r"^constexpr int kProj.*;|^constexpr int kChainAngles.*;", text, re.M))
    const = re.sub(r"//[^;]*?(?=constexpr|$)", "", const)
    fn = re.search(r"^static int project_route\(.*?^}", text, re.M | re.S).group(0)
    return host_build(tmp_path, "route", "#include <algorithm>\n%s\n%s\nextern \"C\" int route(int n, int a, int f) "
                      "{ return project_route(n, a, f); }\n" % (const, fn)).route


def test_projection_tests_run_both_kinds(tmp_path):
    """The sizes of the projection tests lead to the kernels that they compare."""
    route = project_route(tmp_path)
    sizes = next(m.args[1] for m in routes.test_both_projections_agree.pytestmark if m.name == "parametrize")
    for nx, ny, off, A, F, flags in sizes:
        assert (route(1, A, F), route(9, A, F), route(65, A, F)) == (0, 0, 2)
    assert [route(n, 4093, 8) for n in (1, 5, 9, 33)] == [0, 1, 1, 2]
    assert route(1, 180, 8) == route(16, 360, 16) == 0 and route(1024, 360, 16) == 2


@pytest.mark.gpu
@pytest.mark.parametrize("nx, ny, off, flags", [(71, 66, 9, 0), (75, 70, 8, t.FLAG_DFT_FP64)])
def test_all_three_projections_agree(tmp_path, nx, ny, off, flags):
    """One simulation on the vector units, 5 and 9 on the split matrix cores, 33
    on the whole ones: the same far fields bit for bit."""
    route = project_route(tmp_path)
    cfg = routes.small(nx, ny, off, 4093, 8, flags)
    V = seeded_vectors(33, 8, 5)
    V[:, :3] = PHYS_PARAMS[:3]
    T = np.zeros(cfg.farfield_len(), np.float32)
    with t.Context() as c:
        D = {n: c.eval_batch(cfg, V[:n], target=T, want_farfield=True)[1].reshape(n, -1) for n in (33, 9, 5, 1)}
    assert [route(n, 4093, 8) for n in (33, 9, 5, 1)] == [2, 1, 1, 0]
    assert np.abs(D[33]).max() > 0 and np.all(np.isfinite(D[33]))
    for n in (9, 5, 1):
        assert np.array_equal(D[n], D[33][:n]), n


def test_division_by_a_known_divisor(tmp_path):
    """div_known as the kernel has it, compiled for the host: the 32-bit quotient
    itself for every divisor from 1 to 10, but for ties among denormal results."""
    text = open(os.path.join(CSRC, "update_tile.hip")).read()
    line = re.search(r"float div_known\(float a, double r\) \{[^}]*\}", text).group(0)
    use = re.search(r"p\.k = (1\.0 / \(double\)k\[i\]);", text).group(1)
    run = host_build(tmp_path, "div", 'static inline %s\nextern "C" void run(const float* a, const float* k, float* q, long n) {\n'
                     '    for (long i = 0; i < n; ++i) q[i] = div_known(a[i], %s);\n}\n' % (line, use)).run
    rng = np.random.default_rng(5)
    n = 2_000_000
    k = rng.uniform(1, 10, n).astype(np.float32)
    k[:9] = [1, 2, 3, 5, 7, 9, 9.999999, 1.0000001, 10]
    a = rng.integers(0, 2 ** 32, n, dtype=np.uint32).view(np.float32)  # every exponent, NaN and infinities too
    q = np.empty_like(a)
    fp = ctypes.POINTER(ctypes.c_float)
    run(*(x.ctypes.data_as(fp) for x in (a, k, q)), ctypes.c_long(n))
    with np.errstate(all="ignore"):
        want = a / k
    tiny = np.abs(want) < np.finfo(np.float32).tiny
    assert np.array_equal(q[~tiny], want[~tiny], equal_nan=True)
    ulp = np.abs(q[tiny].view(np.int32).astype(np.int64) - want[tiny].view(np.int32))
    assert tiny.sum() > 1000 and ulp.max() <= 1 and (ulp > 0).mean() < 0.01
