"""The FP8 tile kernels write M0 and the LDS-direct load that reads it as two statements (csrc/fp8_gemm.hip): in the built code another instruction
lies between them, and every load's M0 is the one written for it."""
import re

from test_isa_built import _check_m0, _functions, _tool, objects, pytestmark  # noqa: F401


def test_fp8_tile_loads_behind_m0(objects):  # noqa: F811
    checked = 0
    for o in objects:
        for name, code in _functions(_tool("llvm-objdump", "-d", "--mcpu=gfx950", o)).items():
            if "fp8_gemm_kernel" in name and any("global_load_lds_dwordx4" in str(line) for line in code):
                _check_m0(name, code)
                for (_, op, operands, _), (_, follows, _, _) in zip(code, code[1:]):
                    assert not (op == "s_add_u32" and operands[0] == "m0" and follows.startswith("global_load_lds")), name
                checked += 1
    assert checked > 100


def test_rotary_angles_of_a_fetch_are_in_flight_together(objects):  # noqa: F811
    """Behind the K loop of the tiles with rotary embedding: every position is loaded before the first angle, and no wait lies between the angles of one
    fetch (half of the wave's rows; 256-column tiles share the rows between two waves and fetch once).  A position loaded between two angles is waited for,
    and with it every angle ahead of it."""
    checked = set()
    for o in objects:
        for name, code in _functions(_tool("llvm-objdump", "-d", "--mcpu=gfx950", o)).items():
            form = re.match(r"_ZN5llmmm15fp8_gemm_kernelILi(\d+)ELi(\d+)ELi(\d+)ELi[45]ELi(\d)E", name)
            if not form or name.endswith(".kd"):
                continue
            shared, mf = form.group(2) == "256", int(form.group(3)) // 16
            behind = code[max(i for i, c in enumerate(code) if c[1].startswith("v_mfma")) + 1:]
            behind = behind[next(i for i, c in enumerate(behind) if c[1] == "s_barrier"):]
            seen = "".join("L" if op.startswith("global_load_lds") else "g" if op.startswith("global_load") else "w" if op == "s_waitcnt" and "vmcnt" in operands[0] else ""
                           for _, op, operands, _ in behind)
            first, fetch = seen.index("L"), "L" * (mf // 2 * 8)
            assert seen[:first].count("g") == (mf // 2 if shared else mf), (name, seen)
            assert re.findall("L+", seen) == [fetch] * (1 if shared else 2), (name, seen)
            checked.add(form.groups())
    assert len(checked) == 28
