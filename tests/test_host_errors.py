"""The engine's host code where the HIP runtime reports an error, on a double of
that runtime (hip_double.c): no device, kernels do nothing. Each case runs in a
process of its own, which loads the double in the runtime's place."""
import subprocess
import sys

import pytest

from conftest import ROOT

VERSIONS = """
hip_4.2 { global: *; };
hip_4.3 { global: hipGraph*; hipStreamBeginCapture; hipStreamEndCapture; } hip_4.2;
hip_6.0 { global: hipGetDevicePropertiesR0600; } hip_4.3;
"""

SETUP = """
import ctypes as C, sys
hip = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
hip.hip_double_fail.argtypes = [C.c_char_p, C.c_int, C.c_int]
import numpy as np
import n_body_sim_pro_amd as nbx

def engine(n):
    rng = np.random.default_rng(1)
    e = nbx.Engine(n)
    e.upload(rng.normal(size=(n, 3)), np.ones(n))
    return e

def fails(call):
    try:
        call()
    except nbx.NBXError as error:
        return error.status
    return 0

OUT_OF_MEMORY, INVALID_STATE = 2, 3
"""


@pytest.fixture(scope="module")
def double(tmp_path_factory):
    d = tmp_path_factory.mktemp("hip")
    (d / "versions").write_text(VERSIONS)
    lib = d / "libamdhip64.so.7"
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-w", "-Wl,-soname,libamdhip64.so.7",
                    f"-Wl,--version-script={d / 'versions'}", "-o", str(lib),
                    str(ROOT / "tests" / "hip_double.c")], check=True)
    return lib


def run(double, body):
    r = subprocess.run([sys.executable, "-c", SETUP + body, str(double)], cwd=ROOT,
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("algorithm", ["hip_direct_fp64", "hip_direct_fp32"])
@pytest.mark.parametrize("integrator", [0, 1])
def test_advance_reports_what_its_wait_reports(double, algorithm, integrator):
    """All-pairs steps are not waited for one by one: an error of their kernels
    comes with the wait for the whole call."""
    run(double, f"""
e = engine(100)
assert fails(lambda: e.advance("{algorithm}", dt=1e-3, steps=3, integrator={integrator})) == 0
hip.hip_double_fail(b"hipEventSynchronize", 0, 719)
assert fails(lambda: e.advance("{algorithm}", dt=1e-3, steps=3, integrator={integrator})) == INVALID_STATE
""")


@pytest.mark.parametrize("algorithm", ["hip_barnes_hut", "hip_barnes_hut_fp64"])
@pytest.mark.parametrize("n", [5000, 40000])
def test_no_tree_after_an_evaluation_out_of_memory(double, algorithm, n):
    """Whichever allocation of an evaluation fails, there is no tree to report
    on after it: the counts of the last one would not fit the new arrays."""
    run(double, f"""
hip.hip_double_left.restype = C.c_int
k = 0
while True:
    e = engine({n})
    hip.hip_double_fail(b"hipMalloc", k, 2)
    status = fails(lambda: e.compute_force("{algorithm}"))
    if hip.hip_double_left() >= 0:
        break
    assert status == OUT_OF_MEMORY, (k, status)
    assert fails(e.bh_morton) == INVALID_STATE, k
    k += 1
assert k > 15, k
""")


def test_autotune_that_fails_leaves_the_shape(double):
    """The tuner's candidates must not stay behind, whichever upload of their
    items fails, or the graph that times them (which the double does not
    offer)."""
    run(double, """
hip.hip_double_left.restype = C.c_int
e = nbx.Ensemble(np.array([70, 300, 5], dtype=np.uint32))
e.set_tile([2] * 8, 3, 128)
before = e.tile()
k = 0
while True:
    hip.hip_double_fail(b"hipMemcpy", k, 2)
    assert fails(lambda: e.autotune()) != 0, k
    assert e.tile() == before, k
    if hip.hip_double_left() >= 0:
        break
    k += 1
assert k > 5, k
""")
