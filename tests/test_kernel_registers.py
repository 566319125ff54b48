"""What the compiler made of the matmul tiles' registers, read from the built library's kernel descriptions."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "go-inference_amd", "libaq_mi355.so")
READELF = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-readelf")


def _tiles(tmp_path):
    """Template arguments of every qmmh_kernel -> (vector registers, spilled ones)."""
    image, at, found = open(LIB, "rb").read(), 0, {}
    while (at := image.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        count, entry = struct.unpack_from("<Q", image, at + 24)[0], at + 32
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", image, entry)
            name = image[entry + 24:entry + 24 + length]
            entry += 24 + length
            code = image[at + offset:at + offset + size]
            if b"gfx950" not in name or b"qmmh_kernel" not in code:
                continue
            path = tmp_path / "code.o"
            path.write_bytes(code)
            notes = subprocess.run([READELF, "--notes", str(path)], check=True, capture_output=True, text=True).stdout
            for part in notes.split("  - .agpr_count:")[1:]:
                kernel = re.search(r"\.name:\s+\S*qmmh_kernelI((?:Li\d+E)+)E", part)
                if kernel:
                    values = tuple(int(v) for v in re.findall(r"Li(\d+)E", kernel.group(1)))
                    found[values] = tuple(int(re.search(r"\.%s:\s+(\d+)" % key, part).group(1)) for key in ("vgpr_count", "vgpr_spill_count"))
        at += 24
    return found


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_registers_leave_room_for_the_workgroups_that_lds_holds(tmp_path, aqlib):
    tiles = _tiles(tmp_path)
    assert len(tiles) >= 20
    for (bits, mb, nb, wm, wn, stages, elements, group), (registers, spilled) in sorted(tiles.items()):
        name = "%d bit, %d x %d rows and columns, groups of %d" % (bits, wm * mb * 32, wn * nb * 32, group)
        assert spilled == 0, name
        # stages of A and of the packed weights, segments of scales and biases, sums of x
        lds = stages * wm * mb * 4096 + (stages if bits == 8 else 2) * wn * nb * 2048 + 2 * wn * nb * 32 * elements * 2
        lds += wm * mb * 1024 if bits == 4 and mb >= 3 else 0
        by_lds = 160 * 1024 // lds
        by_registers = 512 // ((registers + 7) // 8 * 8) * 4 // (wm * wn)
        assert by_lds >= 1 and by_registers >= by_lds, (name, registers, lds)
