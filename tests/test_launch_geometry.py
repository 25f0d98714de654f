"""What tde_plan reports is what tde_reduce_rms launches, over sizes, types, modes and algorithms
(tests/native/unit_test_launch_geometry.cpp, which stands in for the runtime's launch)."""
import os
import subprocess

from torch_dist_ext_amd import _capi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def test_the_plan_reports_the_launch(tmp_path):
    program = str(tmp_path / "unit_test_launch_geometry")
    library = os.path.dirname(_capi.LIB_PATH)
    build = ["g++", "-O2", "-std=c++17", "-rdynamic", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"), "-I", os.path.join(ROOT, "include"),
             os.path.join(ROOT, "tests", "native", "unit_test_launch_geometry.cpp"), "-o", program, "-L", library, "-ltde_hip",
             "-Wl,-rpath," + library, "-Wl,--allow-shlib-undefined"]
    built = subprocess.run(build, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert built.returncode == 0, built.stdout
    ran = subprocess.run([program], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    print(ran.stdout, flush=True)
    assert ran.returncode == 0, ran.stdout
