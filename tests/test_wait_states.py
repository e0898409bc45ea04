"""Wait states around the inline asm (CPU): in the text of every asm block
whose lane masks are read outside it, and in the machine code of the built
library."""
import glob
import os
import re
import shutil
import subprocess

import pytest
from wait_states import early

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "zeknox_amd", "csrc")
OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"

# lane masks that nothing outside their block reads
UNREAD = {("reduce96_lazy", "s1"), ("reduce128_rare", "b"), ("sub_eps", "b"), ("mul_pow2_lazy", "b")}
UNREAD_ANYWHERE = {"j", "j0", "j1", "bj", "tj", "tj0", "tj1"}
# read two asm blocks on (gl64.h, "carry-out forms"); the library's code is
# checked below
FAR = {("mul128c", "c")}


def asm_blocks():
    """(function, instructions, names of the lane masks written) of every asm block."""
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h"))):
        text = re.sub(r"//[^\n]*", "", open(path).read())
        for m in re.finditer(r"\basm\s*(?:volatile\s*)?\(((?:\s*\"(?:[^\"\\]|\\.)*\")+)\s*:([^;]*?)(?::[^:;]*)?(?::[^:;]*)?\);", text):
            name = re.findall(r"\n__device__[^\n]*?(\w+)\(", text[:m.start()])[-1]
            body = "".join(re.findall(r"\"((?:[^\"\\]|\\.)*)\"", m[1])).replace("\\n\\t", "\n")
            masks = re.findall(r"\[(\w+)\]\s*\"[=+]&?s\"", m[2])
            if masks:
                yield name, body, masks


def test_lane_masks_leave_their_asm_blocks_settled():
    seen = set()
    for name, body, masks in asm_blocks():
        names = sorted(set(re.findall(r"%\[(\w+)\]", body)))
        reg = {n: f"s[{2 * i}:{2 * i + 1}]" if n in masks else f"v[{2 * i}:{2 * i + 1}]" for i, n in enumerate(names)}
        code = re.sub(r"%\[(\w+)\]", lambda m: reg[m[1]], body)
        assert not early(code), name
        for mask in masks:
            if mask in UNREAD_ANYWHERE or (name, mask) in UNREAD | FAR:
                continue
            seen.add((name, mask))
            assert not early(code + f"\nv_cndmask_b32_e64 v900, 0, 1, {reg[mask]}"), (name, mask)
    assert {("reduce96_rare", "c"), ("reduce128_rare2", "b0"), ("reduce128_rare2", "b1"), ("add_sub_lazy2", "b0"),
            ("add_sub_lazy2", "b1"), ("add_sub_lazy2", "k0"), ("add_sub_lazy2", "k1")} <= seen


@pytest.mark.parametrize("text,count", [
    ("v_mad_u64_u32 v[0:1], s[6:7], v4, -1, v[2:3]\nv_writelane_b32 v9, s7, 3", 1),
    ("v_mad_u64_u32 v[0:1], s[6:7], v4, -1, v[2:3]\ns_nop 0\nv_cndmask_b32_e64 v9, 0, 1, s[6:7]", 1),
    ("v_mad_u64_u32 v[0:1], s[6:7], v4, -1, v[2:3]\ns_nop 1\nv_cndmask_b32_e64 v9, 0, 1, s[6:7]", 0),
    ("v_add_co_u32_e32 v1, vcc, v2, v3\nv_mov_b32_e32 v4, v5\nv_addc_co_u32_e32 v6, vcc, v7, v8, vcc", 1),
    ("v_xor_b32_e32 v3, v1, v2\ns_nop 0\nv_mfma_i32_32x32x32_i8 v[16:31], v[0:3], v[4:7], 0", 1),
    ("v_mov_b32_e32 v1, v0\nv_permlane32_swap_b32_e32 v0, v1", 1),
    ("v_mov_b32_e32 v1, v0\ns_nop 1\nv_mov_b32_dpp v2, v1 quad_perm:[1,0,3,2]", 0),
    ("v_mov_b32_e32 v1, v0\nv_readfirstlane_b32 s0, v1", 1),
    ("v_mov_b32_e32 v1, v0\nv_add_u32_e32 v2, v1, v1", 0),
])
def test_the_check_itself(text, count):
    assert len(early(text)) == count


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_built_library(tmp_path):
    lib = os.path.join(ROOT, "zeknox_amd", "libzeknox.so")
    if not os.path.exists(lib):
        pytest.skip("library not built")
    shutil.copy(lib, tmp_path / "lib.so")  # the code objects are written next to it
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    objects = sorted(tmp_path.glob("*gfx950"))
    assert objects
    lines = 0
    for o in objects:
        r = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", o.name], cwd=tmp_path, check=True, capture_output=True, text=True)
        lines += r.stdout.count("\n")
        assert early(r.stdout) == [], o.name
    assert lines > 100000
