"""Static checks of the gfx950 code in the built libllmmm.so, where a kernel is only right or fast by what the compiler makes of it.

The FP16 / BF16 K loop (llmmm_amd/csrc/fp16_gemm.hip) writes its MFMAs and its LDS-direct loads as inline assembly, whose hazards the
compiler does not see: it pads no wait states behind such an MFMA, and does not know that a load reads the M0 that another statement wrote."""
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


# ------------------------------------------------------------------------------------------------ FP16 K loop
def _regs(operand):
    """{('a' | 'v', n)} of a register operand."""
    m = re.fullmatch(r"([av])(?:(\d+)|\[(\d+):(\d+)\])", operand)
    if not m:
        return set()
    lo, hi = (m.group(2), m.group(2)) if m.group(2) else (m.group(3), m.group(4))
    return {(m.group(1), r) for r in range(int(lo), int(hi) + 1)}


def _functions(text):
    """name -> [(address, mnemonic, [operands], branch target or None)]"""
    out, name, base = {}, None, 0
    for line in text.split("\n"):
        m = re.match(r"([0-9a-f]+) <(\w+)>:", line)
        if m:
            base, name = int(m.group(1), 16), m.group(2)
            out[name] = []
            continue
        m = re.match(r"\s+(\S+)(.*?)\s*// ([0-9A-F]+):(.*)", line)
        if m and name:
            t = re.search(r"<%s\+0x([0-9a-f]+)>" % re.escape(name), m.group(4))
            branch = m.group(1).startswith(("s_cbranch", "s_branch"))
            out[name].append((int(m.group(3), 16), m.group(1), [o.strip() for o in m.group(2).split(",")], base + int(t.group(1), 16) if t and branch else None))
    return out


READY = 24  # issue slots after which any MFMA result can be read (16 passes need 19)


def _check_mfma_reads(name, code):
    """No instruction but an MFMA that accumulates in place reads (or overwrites) an MFMA's destination before its result is there, on
    any path: slots since the last MFMA per register, the minimum over all ways into a block."""
    index = {a: i for i, (a, _, _, _) in enumerate(code)}
    starts = sorted({0} | {index[t] for _, _, _, t in code if t is not None} | {i + 1 for i, c in enumerate(code) if c[1].startswith(("s_cbranch", "s_branch"))})
    ends = dict(zip(starts, starts[1:] + [len(code)]))
    entry, work = {0: {}}, [0]
    while work:
        s = work.pop()
        age = dict(entry[s])
        for i in range(s, ends[s]):
            _, op, operands, _ = code[i]
            slots = int(operands[0], 0) + 1 if op == "s_nop" else 1
            if op.startswith("v_mfma"):
                dst = _regs(operands[0])
                assert operands[0] == operands[3], (name, op, operands)
                for o in operands[1:3]:
                    assert not any(age.get(r, READY) < READY for r in _regs(o)), (name, op, operands)
                for back in range(1, 3):  # an operand a VALU instruction writes must be two slots old
                    if i - back >= s and code[i - back][1].startswith("v_") and not code[i - back][1].startswith("v_mfma"):
                        assert not _regs(code[i - back][2][0]) & (_regs(operands[1]) | _regs(operands[2]) | dst), (name, code[i - back], operands)
            else:
                for o in operands:
                    late = [r for r in _regs(o.split(" ")[0]) if age.get(r, READY) < READY]
                    assert not late, "%s: '%s %s' touches MFMA results in flight" % (name, op, ", ".join(operands))
                dst = set()
            age = {r: n + slots for r, n in age.items() if n + slots < READY}
            age.update((r, 0) for r in dst)
        last, succ = code[ends[s] - 1], []
        if last[3] is not None:
            succ.append(index[last[3]])
        if last[1] not in ("s_branch", "s_endpgm") and ends[s] < len(code):
            succ.append(ends[s])
        for t in succ:
            old = entry.get(t)
            new = age if old is None else {r: min(age.get(r, READY), old.get(r, READY)) for r in age.keys() | old.keys()}
            if old is None or new != old:
                entry[t] = new
                work.append(t)


def _check_m0(name, code):
    """Between an M0 written for an LDS-direct load and that load: no other write of M0, no way in or out."""
    targets = {t for _, _, _, t in code if t is not None}
    pending = None
    for a, op, operands, target in code:
        if pending:
            assert a not in targets and target is None, "%s: a block boundary between '%s' and its load" % (name, pending)
            assert operands[0] != "m0", "%s: M0 is written again before the load of '%s'" % (name, pending)
        if op == "s_add_u32" and operands[0] == "m0":
            pending = "%s %s" % (op, ", ".join(operands))
        elif op.startswith("global_load_lds"):
            pending = None
    assert not pending


def test_fp16_loop_hazards(objects):
    path = next(o for o in objects if any("fp16_gemm_kernel" in n for n in _kernels(o)))
    meta = _kernels(path)
    functions = {n: c for n, c in _functions(_tool("llvm-objdump", "-d", path)).items() if re.match(r"_ZN5llmmm\d+fp16_gemm_\w*kernel", n) and not n.endswith(".kd")}
    assert len(functions) == 34 and set(functions) <= set(meta)  # seven tile forms, the hybrid of two: 2 types x 2 layouts; phases: 2 types
    for name, code in functions.items():
        assert int(meta[name]["private_segment_fixed_size"]) == 0 and int(meta[name]["vgpr_spill_count"]) == 0, name
        assert sum(c[1].startswith("v_mfma") for c in code) > 0 and sum(c[1] == "s_add_u32" and c[2][0] == "m0" for c in code) > 0, name
        _check_mfma_reads(name, code)
        _check_m0(name, code)


def test_fp16_split_loop_hazards(objects):
    """The same loop over a share of K (fp16_split_gemm_kernel): its plane stores read the accumulators straight behind it."""
    path = next(o for o in objects if any("fp16_split_gemm_kernel" in n for n in _kernels(o)))
    meta = _kernels(path)
    functions = {n: c for n, c in _functions(_tool("llvm-objdump", "-d", path)).items() if "fp16_split_gemm_kernel" in n and not n.endswith(".kd")}
    assert len(functions) == 12  # three tiles x 2 types x 2 layouts
    for name, code in functions.items():
        assert int(meta[name]["private_segment_fixed_size"]) == 0 and int(meta[name]["vgpr_spill_count"]) == 0, name
        assert sum(c[1].startswith("v_mfma") for c in code) > 0 and sum(c[1] == "s_add_u32" and c[2][0] == "m0" for c in code) > 0, name
        _check_mfma_reads(name, code)
        _check_m0(name, code)


def test_the_checks_see_a_missing_wait_and_a_second_m0_write(objects):
    path = next(o for o in objects if any("fp16_gemm_kernel" in n for n in _kernels(o)))
    name, code = next((n, c) for n, c in _functions(_tool("llvm-objdump", "-d", path)).items() if "fp16_gemm_kernelIDF16_Li64ELi64E" in n and not n.endswith(".kd"))
    with pytest.raises(AssertionError, match="in flight"):
        _check_mfma_reads(name, [(a, "s_nop", ["0"], t) if op == "s_nop" else (a, op, o, t) for a, op, o, t in code])
    i = next(i for i, c in enumerate(code) if c[1] == "s_add_u32" and c[2][0] == "m0")
    with pytest.raises(AssertionError, match="written again"):
        _check_m0(name, code[:i + 1] + [(-1, "s_mov_b32", ["m0", "s3"], None)] + code[i + 1:])
