"""The pipelined prefill kernels of the built library fit as many workgroups on
a CU as their key ranges are planned for (three at head dim 64, two at 96 and
128, one at 256 and with two query blocks a wave), and spill nothing. Read from
the kernels' metadata: a workgroup has one wave per SIMD, a SIMD 512 vector
registers a lane in steps of 8, a CU 160 KiB of LDS."""

import re
import shutil
import subprocess

import pytest

from instinct_amd import _lib

LLVM = "/opt/rocm/llvm/bin"
OBJDUMP, READELF = (shutil.which(x, path=LLVM) or shutil.which(x)
                    for x in ("llvm-objdump", "llvm-readelf"))
PLANNED = {(64, 1): 3, (96, 1): 2, (128, 1): 2, (256, 1): 1, (128, 2): 1}


@pytest.mark.skipif(not (OBJDUMP and READELF), reason="no llvm-objdump or llvm-readelf")
def test_occupancy(tmp_path):
    (tmp_path / "lib.so").symlink_to(_lib.LIBRARY_PATH)
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True,
                   stdout=subprocess.DEVNULL)
    found = {}
    for image in sorted(tmp_path.glob("*gfx950*")):
        if b"prefill_pipe_kernel" not in image.read_bytes():
            continue
        notes = subprocess.run([READELF, "--notes", image.name], cwd=tmp_path, check=True,
                               capture_output=True, text=True).stdout
        for kernel in notes.split("- .agpr_count:")[1:]:
            shape = re.search(r"prefill_pipe_kernelILi(\d+)ELi(\d)ELb(\d)E", kernel)
            if shape:
                field = lambda name: int(re.search(rf"\.{name}: +(\d+)", kernel)[1])  # noqa: B023,E731
                registers, lds = field("vgpr_count"), field("group_segment_fixed_size")
                assert field("private_segment_fixed_size") == field("vgpr_spill_count") == 0
                d, blocks, bf16 = map(int, shape.groups())
                found[d, blocks, bf16] = min(512 // (-(-registers // 8) * 8), 160 * 1024 // lds)
    assert found == {(*key, bf16): n for key, n in PLANNED.items() for bf16 in (0, 1)}
