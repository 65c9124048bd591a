"""The FP8 tile kernels write M0 and the LDS-direct load that reads it as two statements (csrc/fp8_gemm.hip): in the built code another instruction
lies between them, and every load's M0 is the one written for it.  Behind the K loop the rotary angles of a fetch are all in flight together."""
import re

import pytest

from test_isa_built import _check_m0, _functions, _tool, objects, pytestmark  # noqa: F401


@pytest.fixture(scope="module")
def kernels(objects):  # noqa: F811
    """(name, code) of every kernel with FP8 tiles."""
    found = [item for o in objects for item in _functions(_tool("llvm-objdump", "-d", "--mcpu=gfx950", o)).items()]
    return [(n, c) for n, c in found if re.match(r"_ZN5llmmm\d+fp8_gemm_(hybrid_)?kernelI", n) and not n.endswith(".kd")]


def _check_fp8_loads(name, code):
    """Every LDS-direct load reads the M0 that was written for it, with one instruction at least between the two and no way in or out there.
    Returns the number of loads that have more than wait states between."""
    targets = {t for _, _, _, t in code if t is not None}
    write, between, split = None, [], 0
    for address, op, operands, target in code:
        if address in targets or target is not None:
            write = None
        if op.startswith("global_load_lds"):
            assert write is not None, "%s: a load at %x without an M0 of its own" % (name, address)
            assert between, "%s: a load at %x right behind M0" % (name, address)
            split += any(o != "s_nop" for o in between)
            write = None
        elif operands[0] == "m0" and op.startswith("s_"):
            assert write is None, "%s: M0 of the load behind %x is written twice" % (name, address)
            write, between = address, []
        else:
            between.append(op)
    return split


def test_fp8_tile_loads_behind_m0(kernels):
    for name, code in kernels:
        _check_m0(name, code)
        waves_of_32_rows = "hybrid" in name or "ELi32E" in name
        assert (_check_fp8_loads(name, code) > 0) == waves_of_32_rows, name  # their loads have LDS reads or MFMAs behind M0
    assert sum("hybrid" in n for n, _ in kernels) == 18 and len(kernels) == 18 + 289


def test_the_check_sees_a_missing_m0_and_a_missing_wait(kernels):
    code = next(c for n, c in kernels if "hybrid" in n)
    at = [i for i, (_, op, operands, _) in enumerate(code) if op == "s_add_u32" and operands[0] == "m0"]
    with pytest.raises(AssertionError, match="without an M0"):
        _check_fp8_loads("", code[:at[-1]] + code[at[-1] + 1:])
    behind = next(i for i in at if code[i + 1][1] != "s_nop")
    load = next(i for i in range(behind, len(code)) if code[i][1].startswith("global_load_lds"))
    with pytest.raises(AssertionError, match="right behind M0"):
        _check_fp8_loads("", code[:behind + 1] + code[load:])


def test_rotary_angles_of_a_fetch_are_in_flight_together(kernels):
    """Behind the K loop of the tiles with rotary embedding: every position is loaded before the first angle, and no wait lies between the angles of one
    fetch (half of the wave's rows; 256-column tiles share the rows between two waves and fetch once).  A position loaded between two angles is waited for,
    and with it every angle ahead of it."""
    checked = set()
    for name, code in kernels:
        form = re.match(r"_ZN5llmmm15fp8_gemm_kernelILi(\d+)ELi(\d+)ELi(\d+)ELi[45]ELi(\d)E", name)
        if not form:
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
