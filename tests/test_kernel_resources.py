"""Registers of the kernels in the built library, from their code objects'
metadata: what decides how many wavefronts of a kernel share a SIMD (512
VGPRs), and what a kernel moves to memory because it holds more."""

import re
import shutil
import struct
import subprocess

import pytest

from tractography_amd.build import ARCH, LIBRARY

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data):
    at = data.find(MAGIC)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        entry = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            name = data[entry + 24 : entry + 24 + length].decode()
            if ARCH in name and size:
                yield data[at + offset : at + offset + size]
            entry += 24 + length
        at = data.find(MAGIC, at + 1)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    readelf = shutil.which("llvm-readelf", path="/opt/rocm/llvm/bin")
    if readelf is None or not LIBRARY.exists():
        pytest.skip("needs the built library and ROCm's llvm-readelf")
    found = {}
    for i, elf in enumerate(_code_objects(LIBRARY.read_bytes())):
        path = tmp_path_factory.mktemp("code") / f"{i}.elf"
        path.write_bytes(elf)
        notes = subprocess.run([readelf, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for kernel in re.split(r"\n  - \.a", notes)[1:]:
            name = re.search(r"\.name: +(\S+)", kernel[kernel.rindex(".max_flat") :]).group(1)
            found[name] = {k: int(v) for k, v in re.findall(r"\.(\w*gpr\w*count): +(\d+)", kernel)}
    assert len(found) > 100
    return found


def _instance(kernels, name, *arguments):
    """The kernel of that name with these integer template arguments, the
    instance for launches that are never cut short where there are two."""
    pattern = re.compile(name + "I" + "".join(f"Li{a}E" for a in arguments) + "(Lb0E)?E")
    (found,) = [k for k in kernels if pattern.search(k)]
    return kernels[found]


def test_order12_mesh_tracking_spills(kernels):
    # Transport and Diffusion between surfaces, order 12: held to 168 VGPRs
    # they move some to memory; 52 and 40 with the boundary test's answer
    # written to its reference in every branch, which took 5% more time.
    for algorithm in (0, 1):
        k = _instance(kernels, "track_fast_kernel", 0, algorithm, 1, 12, 0)
        assert k["vgpr_count"] <= 168
        assert k["vgpr_spill_count"] <= 40


@pytest.mark.parametrize("model, algorithm, order, vgprs", [
    (1, 0, 8, 72), (1, 1, 8, 72), (1, 2, 8, 96), (1, 3, 8, 96), (0, 0, 12, 168), (0, 1, 12, 168)])
def test_connectomes_of_one_launch(kernels, model, algorithm, order, vgprs):
    # Launches that are never cut short run a kernel without the count of the
    # tracks in flight, which took DTI kernels to 74, 107 and 102 VGPRs and
    # the order-12 Diffusion one to 170: a wavefront per SIMD fewer.
    assert _instance(kernels, "connectome_fast_kernel", model, algorithm, order)["vgpr_count"] <= vgprs
