"""The row kernels (csrc/quant_fp8.hip) on few rows are one pass through code that is not in the instruction cache yet: the rare chunks whose codes need their
quotients go through one piece of code, however many chunks a thread holds."""
import re

from test_isa_built import _functions, _tool, objects, pytestmark  # noqa: F401


def test_the_rare_path_is_there_once(objects):  # noqa: F811
    divisions = {}
    for o in objects:
        for name, code in _functions(_tool("llvm-objdump", "-d", "--mcpu=gfx950", o)).items():
            m = re.match(r"_ZN5llmmm\d+(rmsnorm_quant_row_kernel|planes_add_rmsnorm_quant_kernel)I(DF16b|DF16_|f)Li(\d+)E", name)
            if m and not name.endswith(".kd"):
                divisions[m.groups()] = sum(c[1] == "v_div_fmas_f32" for c in code)
    assert len(divisions) == 36  # two kernels x 3 types x 6 lengths
    # the mean and 1 / sqrt; amax / 448 and four quotients
    assert set(divisions.values()) == {7}, divisions
