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


def test_router_tiles_where_they_are_enough():
    """The frontend's router workgroups: rows up to 64 tokens and where tiles would be few, tiles
    beyond; the published count is the launch's."""
    from hopper_megamoe_basedondeepgemm_amd import _lib, mega
    launch = lambda m, e, h: _lib.load().dgm_frontend_workgroups(m, h, e, 1, _lib.FE_NO_CAST, 1)
    rows = lambda m, e: ((e + 3) // 4) * ((m + 7) // 8 if m >= 64 else (m + 3) // 4)
    tiles = lambda m, e: ((e + 15) // 16) * ((m + 15) // 16)
    for h in (512, 1024, 2048, 3072, 4096):
        for e in (8, 16, 20, 48, 128, 384, 1000):
            for m in (1, 63, 64, 65, 80, 81, 111, 112, 128, 129, 256, 512):
                few = m <= 64 or (h > 1024 and tiles(m, e) <= 64)
                assert launch(m, e, h) == mega.fable_frontend_router_ctas(m, e, h) == (rows if few else tiles)(m, e), (m, e, h)
    assert launch(128, 48, 3072) == 192 and launch(128, 384, 3072) == 192


def test_large_batch_form_runs_one_phase_of_its_formats(tmp_path):
    """Beyond the plain form's tables only launches whose L2 units need no L1 unit of the same launch,
    of the formats that have the form, within its own tables."""
    needs = {(256, 4, 512): 0, (129, 8, 1): 1, (257, 1, 1): 1, (1, 1, 513): 1}
    runs = {(512, 8, 1024, 1, 1, 0, 0): 1, (512, 8, 1024, 1, 6, 0, 0): 1,
            (512, 8, 1024, 1, 3, 0, 0): 0, (512, 8, 1024, 1, 2, 0, 0): 0,      # L2 with its combine
            (512, 8, 1024, 0, 1, 0, 0): 0,                                     # QoQ, NVFP4
            (512, 8, 1024, 1, 1, 1, 0): 0, (512, 8, 1024, 1, 1, 0, 1): 0,      # top-k or frontend in the kernel
            (513, 8, 1024, 1, 1, 0, 0): 0, (512, 8, 1025, 1, 1, 0, 0): 0}      # beyond its tables
    fmt = lambda name, a: f"{name}({', '.join(map(str, a))})"
    assert _eval(tmp_path, [fmt("fused_needs_big", a) for a in needs] + [fmt("fused_big_runs", a) for a in runs]) == \
        list(needs.values()) + list(runs.values())
