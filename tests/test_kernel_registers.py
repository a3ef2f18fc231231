"""Spills of the built kernels, from the metadata of the library's own code
objects (CPU; needs ROCm's binary tools).  A register that lives in scratch is
read back in the step loop, behind the loads that the loop keeps in flight."""

import os
import re
import shutil
import subprocess

import pytest

from fa_rdna3 import _native

TOOLS = "/opt/rocm/llvm/bin"


@pytest.fixture(scope="module")
def spills(tmp_path_factory):
    """{demangled kernel: (spilled vector registers, scratch bytes)} of libfa_mi355x.so."""
    readelf = shutil.which("llvm-readelf", path=TOOLS)
    objcopy = shutil.which("llvm-objcopy", path=TOOLS)
    if not (readelf and objcopy and shutil.which("c++filt")):
        pytest.skip("ROCm's binary tools are not installed")
    tmp = tmp_path_factory.mktemp("objects")
    lib = os.path.join(os.path.dirname(_native.__file__), "libfa_mi355x.so")
    fat = tmp / "fat"
    subprocess.run([objcopy, f"--dump-section=.hip_fatbin={fat}", lib, str(tmp / "out.so")], check=True)
    blob, found = fat.read_bytes(), {}
    # A bundle's code objects are plain ELF images; each starts with the magic.
    starts = [m.start() for m in re.finditer(rb"\x7fELF\x02\x01\x01\x40", blob)]
    for i, at in enumerate(starts):
        one = tmp / f"{i}.o"
        one.write_bytes(blob[at:starts[i + 1] if i + 1 < len(starts) else len(blob)])
        notes = subprocess.run([readelf, "--notes", str(one)], capture_output=True, text=True).stdout
        for kernel in re.split(r"\n\s+- \.a[gr]", notes)[1:]:
            name = re.search(r"\.name:\s+(_Z\S+)", kernel)
            count = re.search(r"\.vgpr_spill_count:\s+(\d+)", kernel)
            scratch = re.search(r"\.private_segment_fixed_size:\s+(\d+)", kernel)
            if name and count and scratch:
                found[name.group(1)] = int(count.group(1)), int(scratch.group(1))
    names = subprocess.run(["c++filt"], input="\n".join(found), capture_output=True, text=True, check=True).stdout
    return dict(zip(names.splitlines(), found.values()))


@pytest.mark.parametrize("kernel", [
    r"bwd_d(kdv|q)_kernel<fa::f32_t,",     # fp32, every head dim and modifier
    r"fwd_kernel<fa::f32_t,",
    r"fwd16_(split_)?kernel<.*, (256|512), 0",
])
def test_kernels_do_not_spill(spills, kernel):
    found = {n: c for n, c in spills.items() if re.search(kernel, n)}
    assert found, sorted(spills)[:5]
    assert not any(c for c, _ in found.values()), {n: c for n, c in found.items() if c[0]}


@pytest.mark.parametrize("kernel,bytes_per_lane", [
    (r"dkdv_roles_kernel<.*, 256, 2>", 256), (r"dkdv16_kernel<.*, 128, 2>", 400), (r"dkdv16_kernel<.*, (32|64), 2>", 0),
])
def test_dropout_backward_keeps_its_step_loop_in_registers(spills, kernel, bytes_per_lane):
    """The sixteen score variants of these kernels took 512 to 576 bytes of
    scratch a lane, most of it read back in the step loop or handed to a
    function there; one variant takes 168 at D = 256, 328 at 128, else none."""
    found = {n: c for n, c in spills.items() if re.search(kernel, n)}
    assert len(found) >= 2 and all(s <= bytes_per_lane for _, s in found.values()), found


@pytest.mark.parametrize("kernel,bytes_per_lane", [(r"dq16_kernel<.*, 128, 1>", 64), (r"dq16_kernel<.*, (32|64), 1>", 0),
                                                   (r"dq16_kernel<.*, (32|64|128), (0|3)>", 64)])
def test_recomputing_dq_is_part_of_its_kernel(spills, kernel, bytes_per_lane):
    """As a function of its own the block took 628 bytes of scratch a lane at
    D = 128 with modifiers; inlined it takes 20."""
    found = {n: c for n, c in spills.items() if re.search(kernel, n)}
    assert len(found) >= 2 and all(s <= bytes_per_lane for _, s in found.values()), found
