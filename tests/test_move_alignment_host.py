"""What alignment a move into a packed copy asks of its source."""
import os
import subprocess

from hiptensor_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_kernels_that_read_any_element_keep_the_declared_alignment(tmp_path):
    """tests/cpp/move_alignment.cpp: a list of layouts, one for each rule that sends one to such a kernel."""
    src, out = os.path.join(ROOT, "tests", "cpp", "move_alignment.cpp"), tmp_path / "move_alignment"
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "include"), "-isystem", "/opt/rocm/include",
                    "-D__HIP_PLATFORM_AMD__", src, "-o", str(out), "-L" + os.path.dirname(_lib.LIB_PATH), "-lhiptensor_amd",
                    "-Wl,-rpath," + os.path.dirname(_lib.LIB_PATH)], check=True, capture_output=True)
    r = subprocess.run([str(out)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip().splitlines()[-1].startswith("ok"), (r.stdout[-2000:], r.stderr)
