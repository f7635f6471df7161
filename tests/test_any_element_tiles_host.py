"""The address arithmetic of the 32/64-bit direct-load tiles that take operands at any element, walked on the CPU."""
import os
import subprocess

from hiptensor_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_requests_lie_inside_and_land_where_they_are_read(tmp_path):
    """tests/cpp/wx_bounds.cpp: random problems planned by the library's planner; every request of the tiles offered for
    them, with the kernel's own address functions (kernels/hd_addr.hpp)."""
    src, out = os.path.join(ROOT, "tests", "cpp", "wx_bounds.cpp"), tmp_path / "wx_bounds"
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "include"), "-isystem", "/opt/rocm/include",
                    "-D__HIP_PLATFORM_AMD__", src, "-o", str(out), "-L" + os.path.dirname(_lib.LIB_PATH), "-lhiptensor_amd",
                    "-Wl,-rpath," + os.path.dirname(_lib.LIB_PATH)], check=True, capture_output=True)
    r = subprocess.run([str(out)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip().splitlines()[-1].startswith("ok"), (r.stdout[-2000:], r.stderr)
