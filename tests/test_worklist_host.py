"""The worklist code of the device library on the host alone
(tests/sanitize/worklist_driver.hip: csrc/device/api.hip compiled without
device code, with stand-ins for the HIP runtime and the class kernels)."""
import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEV = os.path.join(REPO, "libaccint-public_amd", "csrc", "device")

pytestmark = pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not available")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    d = tmp_path_factory.mktemp("worklist")
    obj, exe = str(d / "driver.o"), str(d / "driver")
    for cmd in (["hipcc", "--offload-arch=gfx950", "--offload-host-only", "-O1", "-fPIC", "-std=c++17", "-w",
                 "-I" + os.path.join(REPO, "include"), "-I" + DEV,
                 "-c", os.path.join(REPO, "tests", "sanitize", "worklist_driver.hip"), "-o", obj],
                ["g++", obj, "-pthread", "-o", exe]):
        r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
        assert r.returncode == 0, r.stdout[-4000:]
    return exe


def run(driver, what):
    r = subprocess.run([driver, what], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0 and "worklist driver ok" in r.stdout, r.stdout[-4000:]
    return r.stdout


def test_failed_rebuild_leaves_no_list(driver):
    """A rebuild or a tuning that runs out of memory on the way leaves a handle
    whose calls are refused, not one that runs chunks of one list on the pair
    records of another (or a captured graph on freed ones)."""
    run(driver, "alloc")


def test_chunks_of_divided_kets(driver):
    """The chunks of every run, by class, chain and cap, against their definition
    evaluated entry by entry."""
    assert "divided runs" in run(driver, "cut")


def test_gradient_work_model(driver):
    """The work that the model gives the gradient kernels: what they build (one
    bra and one ket centre raised, closed forms for (ss|ss) and (ps|ss)),
    whatever the order of the quartet's shells."""
    run(driver, "flops")
