"""Host code of the library over a HIP runtime of two devices in host memory
(fake_hip.cpp): what a machine with one GPU, or none, cannot show.  CPU only."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB = os.path.join(ROOT, "cuda-rp_amd", "lib")


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    if not os.path.exists(os.path.join(LIB, "libbubbles_rp.so")):
        import __graft_entry__
        __graft_entry__.build()
    exe = str(tmp_path_factory.mktemp("fake") / "fake_hip")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-rdynamic", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "cuda-rp_amd", "csrc"), "-o", exe,
                    os.path.join(HERE, "fake_hip.cpp"), "-L", LIB, "-lbubbles_rp",
                    f"-Wl,-rpath,{LIB}", "-Wl,--allow-shlib-undefined"],
                   check=True, timeout=120)
    return exe


# devices: read-back, snapshots and restores with the other device current; threads: two
# threads read one handle; slots: a snapshot slot saved again takes no memory; rows: no launch
# is larger in y than the runtime allows
@pytest.mark.parametrize("what", ["devices", "threads", "slots", "rows"])
def test_host_code(fake, what):
    r = subprocess.run([fake, what], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
