"""The staging slots of downloads and uploads, on the host (no GPU): their
header with a runtime of the test's own (io_pool.cpp)."""
import os
import subprocess

import pytest

import minifs_amd as mfs

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(os.path.dirname(mfs.__file__), "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def io_pool(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("io") / "io_pool")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", "-w", "-I", CSRC,
                    "-I", os.path.join(ROCM, "include"), "-o", exe, os.path.join(ROOT, "tests", "io_pool.cpp")],
                   check=True)
    return lambda what: subprocess.run([exe, what], capture_output=True, text=True, timeout=60).stdout.strip()


@pytest.mark.parametrize("what", ["sizes", "two contexts", "many at once", "failed chunk", "no memory",
                                  "no memory, many at once"])
def test_staging_slots(io_pool, what):
    """Transfers of no value to many chunks; a context created, downloading
    and destroyed beside another's download; more transfers than slots; a
    chunk that fails; device or pinned memory for few slots or none, where a
    transfer has to end all the same."""
    assert io_pool(what) == "ok"
