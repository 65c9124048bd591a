"""Static checks of the gfx950 code in the built libllmmm.so, where a kernel is only right or fast by what the compiler makes of it."""
import os
import re
import shutil
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
pytestmark = pytest.mark.skipif(shutil.which(os.path.join(LLVM, "llvm-objdump")) is None, reason="llvm-objdump not available")


def _tool(name, *args):
    return subprocess.run([os.path.join(LLVM, name)] + list(args), stdout=subprocess.PIPE, check=True, text=True).stdout


@pytest.fixture(scope="module")
def objects(tmp_path_factory):
    """Paths of the code objects in the library's offload bundles."""
    lib = open(os.path.join(ROOT, "llmmm_amd", "libllmmm.so"), "rb").read()
    out, at = [], lib.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", lib, at + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", lib, entry)
            if b"gfx950" in lib[entry + 24:entry + 24 + length] and size:
                path = str(tmp_path_factory.mktemp("co") / "code.elf")
                open(path, "wb").write(lib[at + offset:at + offset + size])
                out.append(path)
            entry += 24 + length
        at = lib.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 1)
    assert out
    return out


def _kernels(path):
    """name -> {vgpr_count, private_segment_fixed_size, ...} of a code object's metadata."""
    out = {}
    for part in _tool("llvm-readelf", "--notes", path).split("  - .agpr_count:")[1:]:
        fields = dict(re.findall(r"\.(\w+): +(\S+)", "    .agpr_count:" + part))
        out[fields["name"]] = fields
    return out


def test_rotary_kernel_behind_planes_keeps_five_waves(objects):
    """10240 columns at M = 128 are 1280 workgroups of one wave per SIMD: five of them on every CU at once, or a second round."""
    found = {n: k for o in objects for n, k in _kernels(o).items() if "fp8_planes_qk_norm_rope_kernel" in n}
    assert len(found) == 2
    for n, k in found.items():
        assert int(k["vgpr_count"]) <= 96 and int(k["private_segment_fixed_size"]) == 0, (n, k)
