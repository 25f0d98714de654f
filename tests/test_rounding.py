"""The row kernels' reciprocals, roots and quotients against the plain IEEE operations, on the host: every mantissa, every
approximation that the hardware's instructions may start them from (tests/native/unit_test_rounding.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")


def test_every_rounding_is_the_ieee_operations(tmp_path):
    program = str(tmp_path / "unit_test_rounding")
    # fused multiply-adds only where they are written, as in the kernels' build; in hardware where the host has them
    fma = ["-Xarch_host", "-mfma"] if " fma " in open("/proc/cpuinfo").read() else []
    build = [HIPCC, "-x", "hip", "--offload-host-only", "--offload-arch=gfx950", "-O2", "-std=c++17", "-ffp-contract=off", "-pthread", *fma,
             "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "torch_dist_ext_amd", "csrc"),
             os.path.join(ROOT, "tests", "native", "unit_test_rounding.cpp"), "-o", program]
    built = subprocess.run(build, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert built.returncode == 0, built.stdout
    ran = subprocess.run([program], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    print(ran.stdout, flush=True)
    assert ran.returncode == 0, ran.stdout
