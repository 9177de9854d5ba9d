"""The launch shapes of the implicit pass.  The size rule
(koral-zig_amd/csrc/kz_sim_dev.h), evaluated by the compiler: the width of a
batch's persistent launches, which the tuner varies, does not move the size
from which a grid's first rung is launched at two waves per SIMD.  And the
built library holds the kernels of the shapes that calls reach, no others."""
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


def test_no_kernel_without_a_caller():
    names = (CSRC.parent / "lib" / "libkz_hip.so").read_bytes()
    for cells in (b"9GridCells", b"10MultiCells"):
        for shape in (b"11k_imp_rung0I", b"19k_imp_rung0_persistI", b"20k_imp_ladder_persistI"):
            assert shape + cells in names, (shape, cells)
    assert b"19k_imp_rung0_persistI10BatchCells" in names
    assert b"11k_imp_rung0I10BatchCells" not in names  # batches run the persistent launches only
