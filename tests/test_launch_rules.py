"""The host's rules about launches of the persistent kernel (csrc/dgm_fused.hpp), compiled for the CPU."""
import subprocess

import pytest

from hopper_megamoe_basedondeepgemm_amd.build import CSRC


def _eval(tmp_path, exprs):
    """The integer values of C++ expressions over dgm_fused.hpp."""
    src = tmp_path / "rules.cpp"
    src.write_text('#include <stdio.h>\n#include "dgm_fused.hpp"\nint main() {\n'
                   + "".join(f'  printf("%d\\n", (int)({e}));\n' for e in exprs) + "}\n")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{CSRC}", str(src), "-o",
                    str(tmp_path / "rules")], check=True)
    out = subprocess.run([str(tmp_path / "rules")], check=True, capture_output=True, text=True).stdout
    return [int(v) for v in out.split()]


def test_launches_that_wait_on_other_workgroups(tmp_path):
    """The whole layer, L2 with its combine, and anything with the in-kernel frontend; not L1 alone
    (phases 1) nor L2 before a combine launch (2 | 4). A cooperative launch is made for these only."""
    cases = {(1, 0): 0, (6, 0): 0, (2, 0): 1, (3, 0): 1, (1, 1): 1, (3, 1): 1}
    assert _eval(tmp_path, [f"fused_launch_waits({p}, {f})" for p, f in cases]) == list(cases.values())
