"""Two facts that other tests restate in Python, held to the kernel sources
themselves: the rule that picks a far-field projection, and the reference
stage's division by a known kappa."""
import ctypes
import os
import re
import subprocess

import numpy as np

import test_projection_routes as routes

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tomography_amd", "csrc")


def test_projection_rule_is_the_dispatch_s_own():
    """The restated rule against launch_project's expressions and constants."""
    text = open(os.path.join(CSRC, "kernels.hip")).read()
    const = {k: int(v) for k, v in re.findall(r"\b(kChain\w+|kProj\w+) = (\d+)\b", text)}
    const["kProjAngles"] = 32 * const["kProjAngleTiles"]
    body = text[text.index("hipError_t launch_project("):]
    rule = dict(re.findall(r"const int (chain|mfma) = ([^;]+);", body))
    cond = re.search(r"if \((chain < [^{]+)\) \{", body).group(1)

    def on_matrix_cores(n_sims, n_angles, n_freq):
        env = dict(const, n_sims=n_sims, n_angles=n_angles, n_freq=n_freq)
        for name in ("chain", "mfma"):
            env[name] = eval(rule[name].replace("/", "//"), {}, env)
        return not eval(cond.replace("/", "//"), {}, env)

    picks = set()
    for n in (1, 2, 8, 9, 31, 32, 33, 64, 65, 127, 128, 200, 256, 257, 1024, 4000):
        for A in (1, 24, 100, 180, 360, 720, 723, 1921, 4096):
            for F in (1, 3, 8, 16, 32):
                assert on_matrix_cores(n, A, F) == routes.on_matrix_cores(n, A, F), (n, A, F)
                picks.add(on_matrix_cores(n, A, F))
    assert picks == {True, False}


def test_division_by_a_known_divisor(tmp_path):
    """div_known as the kernel has it, compiled for the host: the 32-bit quotient
    itself for every divisor from 1 to 10, but for ties among denormal results."""
    text = open(os.path.join(CSRC, "update_tile.hip")).read()
    line = re.search(r"float div_known\(float a, double r\) \{[^}]*\}", text).group(0)
    use = re.search(r"p\.k = (1\.0 / \(double\)k\[i\]);", text).group(1)
    src = tmp_path / "div.cpp"
    src.write_text('static inline %s\nextern "C" void run(const float* a, const float* k, float* q, long n) {\n'
                   '    for (long i = 0; i < n; ++i) q[i] = div_known(a[i], %s);\n}\n' % (line, use))
    lib = tmp_path / "div.so"
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-shared", "-fPIC", str(src), "-o", str(lib)], check=True)
    run = ctypes.CDLL(str(lib)).run
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
