"""The size rule of the implicit pass (koral-zig_amd/csrc/kz_sim_dev.h),
evaluated by the compiler: the width of a batch's persistent launches, which
the tuner varies, does not move the size from which a grid's first rung is
launched at two waves per SIMD."""
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "koral-zig_amd" / "csrc"


@pytest.mark.parametrize("width", [2, 4, 8])
def test_wide_rule_is_not_the_batch_width(width, tmp_path):
    src = tmp_path / "rule.hip"
    src.write_text('#include "kz_sim_dev.h"\n'
                   "static_assert(wide_cells(256) == 196608, \"three cells for every lane of 1024 SIMDs\");\n"
                   "static_assert(wide_cells(64) * 4 == wide_cells(256), \"\");\n")
    subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-std=c++17", "--cuda-host-only", "-fsyntax-only",
                    f"-DKZ_PERSIST_PER_CU={width}", "-I", str(CSRC), str(src)], check=True)
