"""The search of the compiled assembly for spills ahead of an exec restore
(koral-zig_amd/asmcheck.py): what it must report, what it must let pass, and
that a build with a finding leaves no library behind."""
import importlib.util
from pathlib import Path

import pytest

PKG = Path(__file__).resolve().parent.parent / "koral-zig_amd"


def _load(name):
    spec = importlib.util.spec_from_file_location("kz_" + name, PKG / f"{name}.py")
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


asmcheck = _load("asmcheck")

HEAD = "_Z1kv:\n\ts_load_dword s0, s[4:5], 0x0\n"
RESTORE = "\ts_or_b64 exec, exec, s[0:1]\n\tv_add_f64 v[0:1], v[2:3], v[4:5]\n"
MASK = "\tv_readlane_b32 s0, v63, 4\n\tv_readlane_b32 s1, v63, 5\n"
LOST = {
    "accumulator": ".LBB0_7:                               ; %Flow\n" + MASK + "\tv_accvgpr_write_b32 a12, v7\n" + RESTORE,
    "accumulator-read": ".LBB0_7:\n" + MASK + "\tv_accvgpr_read_b32 v7, a12\n" + RESTORE,
    "scratch": ".LBB0_7:\n" + MASK + "\tscratch_store_dwordx2 off, v[6:7], off offset:16 ; 8-byte Folded Spill\n" + RESTORE,
    "copy": ".LBB0_7:\n" + MASK + "\tv_mov_b32_e32 v9, v7\n" + RESTORE,
    # the block behind a loop has no label: no lane is on before its restore
    "loop-exit": ".LBB0_6:\n\ts_andn2_b64 exec, exec, s[2:3]\n\ts_cbranch_execnz .LBB0_6\n; %bb.7:\n" + MASK +
                 "\tv_accvgpr_write_b32 a12, v7\n" + RESTORE,
    "other-side": ".LBB0_7:                               ; %Flow\n" + MASK +
                  "\tv_accvgpr_write_b32 a12, v7\n\ts_or_saveexec_b64 s[0:1], s[0:1]\n\ts_xor_b64 exec, exec, s[0:1]\n",
    "behind-whole-wave": ".LBB0_7:\n\ts_or_saveexec_b64 s[8:9], -1\n\tv_accvgpr_read_b32 v63, a3\n"
                         "\ts_mov_b64 exec, s[8:9]\n" + MASK + "\tv_accvgpr_write_b32 a12, v7\n" + RESTORE,
}
SOUND = {
    "after": ".LBB0_7:\n" + MASK + RESTORE + "\tv_accvgpr_write_b32 a12, v7\n",
    "whole-wave": ".LBB0_7:\n\ts_or_saveexec_b64 s[8:9], -1\n\tv_accvgpr_read_b32 v63, a3\n\ts_mov_b64 exec, s[8:9]\n" +
                  MASK + RESTORE,
    # a branch's own code in one block with the rejoining lanes
    "branch-body": ".LBB0_7:\n\tv_mov_b32_e32 v4, v7\n\tglobal_store_dwordx2 v[2:3], v[4:5], off\n" + RESTORE,
    "no-rejoin": ".LBB0_7:\n\tv_accvgpr_write_b32 a12, v7\n\ts_cbranch_execz .LBB0_9\n; %bb.8:\n" + RESTORE,
}


@pytest.mark.parametrize("name", sorted(LOST))
def test_reported(name):
    found = asmcheck.lost_lanes(HEAD + LOST[name])
    assert len(found) == 1 and found[0][0] == "_Z1kv" and found[0][1] in (".LBB0_7", "%bb.7"), found


@pytest.mark.parametrize("name", sorted(SOUND))
def test_let_pass(name):
    assert asmcheck.lost_lanes(HEAD + SOUND[name]) == []


def test_build_is_refused(tmp_path, monkeypatch):
    """compile_hip searches the assembly of every source; with a finding it
    raises and writes no library, without one it links."""
    build = _load("build")
    srcs = []
    for k in ("one", "two"):
        srcs.append(tmp_path / f"{k}.hip")
        srcs[-1].write_text(f"#include <hip/hip_runtime.h>\n__global__ void kernel_{k}(double *x) {{ *x = 1.0; }}\n")
    monkeypatch.setattr(build, "HIP_SOURCES", srcs)
    texts = []

    def plant(text):
        texts.append(text)
        return real(text + "\n" + HEAD + LOST["accumulator"])

    real = build.asmcheck.lost_lanes
    monkeypatch.setattr(build.asmcheck, "lost_lanes", plant)
    out = tmp_path / "lib.so"
    with pytest.raises(RuntimeError, match="exec restore"):
        build.compile_hip(out)
    assert not out.exists()
    assert len(texts) == 2 and all("kernel_" + k in t and "gfx950" in t for k, t in zip(("one", "two"), texts))
    monkeypatch.setattr(build.asmcheck, "lost_lanes", real)
    build.compile_hip(out)
    assert out.exists()
