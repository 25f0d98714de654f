"""No kernel of the built library keeps anything in scratch memory: what its own metadata says."""
import os
import re
import subprocess

from torch_dist_ext_amd import _capi

READELF = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "lib", "llvm", "bin", "llvm-readelf")
EM_AMDGPU = 224


def _kernels(tmp_path):
    """(name, scratch bytes, spilled vector registers, spilled scalar registers) of every kernel: the library holds one code object per source."""
    library = open(_capi.LIB_PATH, "rb").read()
    at, found = library.find(b"\x7fELF", 4), []
    while at != -1:
        if int.from_bytes(library[at + 18: at + 20], "little") == EM_AMDGPU:
            one = tmp_path / ("code_object_%d" % at)
            one.write_bytes(library[at:])
            notes = subprocess.run([READELF, "--notes", str(one)], stdout=subprocess.PIPE, stderr=subprocess.DEVNULL, text=True).stdout
            one.unlink()
            for kernel in re.split(r"^  - ", notes, flags=re.M)[1:]:
                name = re.search(r"^    \.name: +(\S+)", kernel, re.M)
                if name:
                    found.append((name.group(1), *(int(re.search(r"\.%s: +(\d+)" % k, kernel).group(1))
                                                   for k in ("private_segment_fixed_size", "vgpr_spill_count", "sgpr_spill_count"))))
        at = library.find(b"\x7fELF", at + 4)
    return found


def test_no_kernel_touches_scratch(tmp_path):
    kernels = _kernels(tmp_path)
    assert len([k for k in kernels if "row_kernel" in k[0]]) > 500
    assert [k for k in kernels if any(k[1:])] == []


def test_owned_rows_of_two_vectors_keep_eight_wavefronts(tmp_path):
    """Owned rows of eight partials with two vectors per thread read two streams for most rows and need every wavefront they can get: 64 registers."""
    library = open(_capi.LIB_PATH, "rb").read()
    at, found = library.find(b"\x7fELF", 4), {}
    while at != -1:
        if int.from_bytes(library[at + 18: at + 20], "little") == EM_AMDGPU:
            one = tmp_path / ("code_object_%d" % at)
            one.write_bytes(library[at:])
            notes = subprocess.run([READELF, "--notes", str(one)], stdout=subprocess.PIPE, stderr=subprocess.DEVNULL, text=True).stdout
            one.unlink()
            for kernel in re.split(r"^  - ", notes, flags=re.M)[1:]:
                name = re.search(r"^    \.name: +(\S*row_kernelINS_\S+ELi8ELi2ELi\dELb\dELi3E\S+)", kernel, re.M)   # partials, vectors, quant, rows too, form
                if name:
                    found[name.group(1)] = int(re.search(r"\.vgpr_count: +(\d+)", kernel).group(1))
        at = library.find(b"\x7fELF", at + 4)
    assert len(found) >= 2 * 3 * 7
    assert {k: v for k, v in found.items() if v > 64} == {}
