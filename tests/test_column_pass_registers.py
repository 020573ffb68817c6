"""No register of the sparse column pass (d = 32) is reloaded inside its loop over tiles: such a reload waits for every load in
flight, and so for the tiles on their way into LDS.  Looks at the device assembly of the kernels (a few seconds of compilation)."""
import os
import re

from spion_amd import build


def _tile_loops(asm):
    """{kernel: [lines of each innermost loop with matrix instructions]}"""
    found = {}
    for name, body in re.findall(r"^(_Z\w+):.*?$(.*?)^\.Lfunc_end", asm, re.M | re.S):
        lines, at, loops = body.split("\n"), {}, []
        for n, line in enumerate(lines):
            if m := re.match(r"(\.LBB\w+):", line):
                at[m.group(1)] = n
            elif (m := re.search(r"s_c?branch\w*\s+(\.LBB\w+)", line)) and m.group(1) in at:
                loops.append((at[m.group(1)], n))
        inner = [a for a in loops if not any(b != a and a[0] <= b[0] and b[1] <= a[1] for b in loops)]
        parts = [lines[a:b + 1] for a, b in inner]
        found[name] = [part for part in parts if any("v_mfma" in x for x in part)]
    return found


def test_no_reload_in_the_tile_loops(tmp_path):
    layouts = ("true, false", "false, false", "true, true")  # row-major, feature-major, strided heads
    kernels = [f"(const void*)&tile_bwd_col_kernel<32, {w}, {x}>" for w in (1, 2, 4, 8) for x in layouts]
    src = tmp_path / "columns.hip"
    src.write_text(f'#include "{build.CSRC}/common.h"\n#include "{build.CSRC}/tile_kernels.h"\nusing namespace spion;\n'
                   f'const void* const kernels[] = {{{", ".join(kernels)}}};\n')
    asm = open(build.emit_device_asm(str(src), os.path.join(tmp_path, "columns.s"))).read()
    loops = {k: v for k, v in _tile_loops(asm).items() if "tile_bwd_col_kernel" in k}
    assert len(loops) == len(kernels)
    for name, parts in loops.items():
        assert len(parts) == 2, (name, len(parts))  # the walk on split operands, the one on whole ones
        assert not [x for part in parts for x in part if "scratch_load" in x], name
