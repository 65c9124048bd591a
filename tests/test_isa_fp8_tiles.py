"""The FP8 tile kernels write M0 and the LDS-direct load that reads it as two statements (csrc/fp8_gemm.hip): in the built code another instruction
lies between them, and every load's M0 is the one written for it."""
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
