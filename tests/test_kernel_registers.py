"""What the compiler made of the registers of the matmul tiles and of the expert blocks, read from the built library's kernel descriptions."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "go-inference_amd", "libaq_mi355.so")
READELF = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-readelf")


def _kernels(tmp_path, kernel_name, *keys):
    """Template arguments of every kernel of that name -> what its description says under the keys."""
    image, at, found = open(LIB, "rb").read(), 0, {}
    while (at := image.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        count, entry = struct.unpack_from("<Q", image, at + 24)[0], at + 32
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", image, entry)
            name = image[entry + 24:entry + 24 + length]
            entry += 24 + length
            code = image[at + offset:at + offset + size]
            if b"gfx950" not in name or kernel_name.encode() not in code:
                continue
            path = tmp_path / "code.o"
            path.write_bytes(code)
            notes = subprocess.run([READELF, "--notes", str(path)], check=True, capture_output=True, text=True).stdout
            for part in notes.split("  - .agpr_count:")[1:]:
                kernel = re.search(r"\.name:\s+\S*%sI((?:Li\d+E)+)E" % kernel_name, part)
                if kernel:
                    values = tuple(int(v) for v in re.findall(r"Li(\d+)E", kernel.group(1)))
                    found[values] = tuple(int(re.search(r"\.%s:\s+(\d+)" % key, part).group(1)) for key in keys)
        at += 24
    return found


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_registers_leave_room_for_the_workgroups_that_lds_holds(tmp_path, aqlib):
    tiles = _kernels(tmp_path, "qmmh_kernel", "vgpr_count", "vgpr_spill_count")
    assert len(tiles) >= 20
    for (bits, mb, nb, wm, wn, stages, elements, group), (registers, spilled) in sorted(tiles.items()):
        name = "%d bit, %d x %d rows and columns, groups of %d" % (bits, wm * mb * 32, wn * nb * 32, group)
        assert spilled == 0, name
        # stages of A and of the packed weights, segments of scales and biases, sums of x, factors of the rows (two kernels of 8 bit read
        # them from memory)
        lds = stages * wm * mb * 4096 + (stages if bits == 8 else 2) * wn * nb * 2048 + 2 * wn * nb * 32 * elements * 2
        lds += wm * mb * 1024 if bits == 4 and mb >= 3 else 0
        lds += wm * mb * 128 if not (bits == 8 and mb == 2 and wm * wn == 4) else 0
        by_lds = 160 * 1024 // lds
        by_registers = 512 // ((registers + 7) // 8 * 8) * 4 // (wm * wn)
        assert by_lds >= 1 and by_registers >= by_lds, (name, registers, lds)


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_expert_blocks_leave_room_for_three_workgroups(tmp_path, aqlib):
    """aq_qmm_routes.hip: three workgroups of four wavefronts to a CU, two in groups of 32."""
    blocks = _kernels(tmp_path, "qmmr_kernel", "vgpr_count", "vgpr_spill_count", "group_segment_fixed_size")
    assert sorted(blocks) == [(32,), (64,), (128,)]
    for (group,), (registers, spilled, lds) in blocks.items():
        workgroups = 2 if group == 32 else 3
        assert spilled == 0 and 512 // ((registers + 7) // 8 * 8) >= workgroups and 160 * 1024 // lds >= workgroups, (group, registers, lds)
