"""What the compiler made of the persistent kernel (csrc/program.hip), read from the assembly of this tree's own source.

The kernel keeps values that are derived from the lane in registers across loops and branches that mask lanes off.  The
compiler sees one flow of control for the wave, so where it splits such a register's live range it may copy the register
under a mask.  Inside a masked region that is harmless: both copies touch the same lanes, and the others keep the register
they had.  It is wrong only where a region is left: a copy that stands in the block where the lanes come back, but before the
instruction that brings them back, leaves the other lanes' values behind (and likewise one behind the instruction that masks
lanes off, where the block goes on to code that runs for all).  Neither may be in the kernel, nor a register spilled to memory."""
import os
import re
import subprocess

import pytest

from dldt_amd import build

VECTOR = re.compile(r"(v_|scratch_|buffer_|global_|ds_|flat_)")
LANE = ("v_readlane_b32", "v_writelane_b32")        # scalar registers kept in lanes: these ignore the mask


def masked_writes(lines):
    """(line number, what) of every vector instruction in front of the end of a mask, or behind its start, in one block"""
    found, vector, narrowed, defs = [], [], None, {}
    for n, line in enumerate(lines, 1):
        s = line.strip()
        if re.match(r"\.LBB\d+_\d+:", line) or s.startswith("; %bb."):
            vector, narrowed, defs = [], None, {}
            continue
        if not s or s[0] in ";.":
            continue
        op, _, rest = s.partition(" ")
        target = rest.split(",")[0].strip()
        if VECTOR.match(op):
            if op not in LANE:
                vector.append(s)
                if narrowed:
                    found.append((n, "%s behind %s" % (s, narrowed)))
            continue
        narrows = op in ("s_and_saveexec_b64", "s_andn2_saveexec_b64") or (op in ("s_and_b64", "s_andn2_b64", "s_xor_b64") and target == "exec")
        if op == "s_mov_b64" and target == "exec":      # the mask of a branch computed beside its saved copy
            narrows = defs.get(rest.split(",")[1].strip()) == "s_and_b64"
        if narrows:
            narrowed = s
        elif target == "exec" or op == "s_or_saveexec_b64":
            if vector:
                found.append((n, "%s in front of %s" % (vector[0], s)))
            narrowed = None
        defs[target] = op
    return found


@pytest.mark.parametrize("text,count", [
    ("; %bb.1:\n s_or_b64 exec, exec, s[4:5]\n v_mov_b32_e32 v1, v2", 0),
    ("; %bb.1:\n v_readlane_b32 s6, v245, 3\n s_or_b64 exec, exec, s[4:5]", 0),
    ("; %bb.1:\n v_mov_b32_e32 v1, v2\n s_or_b64 exec, exec, s[4:5]", 1),
    (".LBB0_3:\n v_accvgpr_read_b32 v1, a2\n s_or_saveexec_b64 s[2:3], s[2:3]", 1),
    (".LBB0_3:\n v_mov_b32_e32 v1, v2\n s_mov_b64 exec, s[2:3]", 1),
    (".LBB0_3:\n v_cmp_gt_i32_e32 vcc, s1, v1\n s_and_b64 s[2:3], s[4:5], vcc\n s_mov_b64 exec, s[2:3]\n s_cbranch_execz .LBB0_4", 0),
    (".LBB0_3:\n s_andn2_b64 exec, exec, s[8:9]\n v_mov_b32_e32 v1, v2\n s_cbranch_execnz .LBB0_3", 1),
    (".LBB0_3:\n v_cmp_gt_i32_e32 vcc, s1, v1\n s_and_saveexec_b64 s[2:3], vcc\n s_cbranch_execz .LBB0_4\n; %bb.4:\n v_mov_b32_e32 v1, v2", 0),
])
def test_the_reading_of_the_assembly(text, count):
    assert len(masked_writes(text.splitlines())) == count


def test_no_register_is_copied_where_a_mask_of_the_persistent_kernel_ends(tmp_path):
    out = tmp_path / "program.s"
    subprocess.run([build.HIPCC] + build.FLAGS + ["-x", "hip", "--offload-device-only", "-S", os.path.join(build.CSRC, "program.hip"), "-o", str(out)],
                   check=True, capture_output=True)
    text = out.read_text()
    found = [m.start() for m in re.finditer(r"^_ZN\S*program_kernel\S*:", text, re.M)]
    assert len(found) == 3                                          # feature maps, encoders, both
    for start in found:
        kernel = text[start:]
        kernel = kernel[:kernel.index(".end_amdhsa_kernel")]
        lines = kernel.splitlines()
        assert sum("exec, exec" in line for line in lines) > 40     # the masks are there to be read
        assert masked_writes(lines) == []
        assert re.search(r"\.amdhsa_private_segment_fixed_size 0\b", kernel)
    assert set(re.findall(r"\.vgpr_spill_count: *(\d+)", text)) == {"0"}
