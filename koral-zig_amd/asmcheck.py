"""Search of the compiled gfx950 assembly for spills that lose lanes.

Where lanes rejoin, a block begins by widening the exec mask (`s_or_b64 exec`
at the end of a branch or loop, `s_or_saveexec_b64` between the two sides of a
branch).  When the mask's own scalar pair has been spilled, it is read back
there first, and the compiler can then place a vector spill, reload or copy
ahead of the restore: the lanes that come back keep a stale value.  Two builds
of the ladder kernel did so and gave wrong rungs for one cell in ten.  Neither
the source nor a compiler option rules it out, so every build is searched.

A spill ahead of a restore is reported even where the lanes that come back
would never read it.  A register copy is reported only where no other vector
instruction stands beside it: a branch's own code that ends in the restore
holds copies too.
"""
import re

_FUNCTION = re.compile(r"([A-Za-z_]\w*):")
_BLOCK = re.compile(r"(\.LBB\w+):|; (%bb\.\d+):")
_RESTORE = re.compile(r"s_or_b64 exec, exec, |s_or_saveexec_b64 ")
_WHOLE_WAVE = re.compile(r"s_or_saveexec_b64 (s\[\d+:\d+\]), -1$")
_VECTOR = re.compile(r"(v_|global_|ds_|scratch_|buffer_|flat_)")
_LANE = re.compile(r"v_(readlane|writelane|readfirstlane)_")  # the same under any mask
_SPILL = re.compile(r"v_accvgpr_|scratch_|buffer_(load|store)_\w+ .*\boff, s\[0:3\]")
_COPY = re.compile(r"v_mov_b(32|64)_|v_pk_mov_b32")  # also a constant formed anew


def _head(lines):
    """The vector instructions of a block ahead of its exec restore, [] if it
    has none or does not begin with scalar work and a restore."""
    found, whole = [], None
    for line in lines:
        if whole:  # all lanes are on: what stands here loses none
            if line == f"s_mov_b64 exec, {whole}":
                whole = None
            continue
        m = _WHOLE_WAVE.match(line)
        if m:
            whole = m.group(1)
        elif _RESTORE.match(line):
            return found
        elif "exec" in line or line.startswith("s_cbranch"):
            return []
        elif _VECTOR.match(line) and not _LANE.match(line):
            found.append(line)
    return []


def lost_lanes(text):
    """[(function, block, instructions)] of the blocks in an assembly listing
    whose spills, reloads or copies stand ahead of the exec restore."""
    found = []
    function, block, lines = None, None, []

    def close():
        head = _head(lines)
        spills = [x for x in head if _SPILL.match(x)]
        if not spills and head and all(_COPY.match(x) for x in head):
            spills = head
        if spills:
            found.append((function, block, spills))

    for raw in text.splitlines():
        m = _BLOCK.match(raw)
        f = None if m else _FUNCTION.match(raw)
        if m or f:
            close()
            lines = []
            block = (m.group(1) or m.group(2)) if m else "entry"
            function = f.group(1) if f else function
            continue
        line = " ".join(raw.split(";")[0].split())
        if line and not line.startswith("."):
            lines.append(line)
    close()
    return found
