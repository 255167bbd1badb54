"""The wait states gfx950 asks for between a vector instruction's write and a later vector read, in the built kernels.
The compiler inserts them in its own code but does not look inside inline assembly (the wave decoder's literal loop), so
the library's disassembly is checked:

  an SGPR or vcc written by a vector instruction (compare, lane read, carry), then read by one: 2 wait states, or 4
  where it is a lane select
  exec written by a vector compare (v_cmpx), then a lane read or write: 4
  a VGPR, then a lane read of it: 1
  a VGPR written in part (SDWA dst_sel other than DWORD), then a vector read of it: 1

An instruction is one wait state, s_nop N is N + 1. Straight-line order; runs without a GPU."""
import os
import re
import shutil
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "panvram_amd", "libpanvram_amd.so")
BIN = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
LANE = ("v_readlane", "v_readfirstlane", "v_writelane")
REG = re.compile(r"\b([sv])(?:(\d+)\b|\[(\d+):(\d+)\])|\b(vcc|exec)\b")


def _regs(text):
    """The registers an operand names: {"s5", "v64", "vcc", ...}."""
    out = set()
    for kind, one, lo, hi, name in REG.findall(text):
        if name:
            out.add(name)
        else:
            out.update(f"{kind}{i}" for i in (range(int(lo), int(hi) + 1) if lo else (int(one),)))
    return out


def _access(op, args):
    """(registers written, registers read) of a vector instruction, as far as the rules above need them."""
    if op.startswith(("global_", "flat_", "scratch_", "buffer_", "ds_")):
        return set(), set()
    two = bool(re.match(r"v_(add|sub|subrev|addc|subb|subbrev)_co_|v_div_scale|v_mad_[iu]64_|v_swap", op))
    k = 2 if two else 1
    wrote = set().union(*(_regs(a) for a in args[:k]))
    read = set().union(set(), *(_regs(a) for a in args[k:]))
    if op.startswith("v_cmpx"):
        wrote.add("exec")
    if op.startswith("v_writelane"):
        read |= wrote
    return wrote, read


def violations(lines):
    found, kernel = [], ""
    made = {}                                  # register -> (state count after its write, partial VGPR write)
    now = 0
    for line in lines:
        if line.endswith(">:"):
            kernel, made = line, {}
            continue
        body = line.split("//")[0].strip()
        if not body:
            continue
        op, _, rest = body.partition(" ")
        now += 1
        if op == "s_nop":
            now += int(rest, 0)
        if not op.startswith("v_"):
            if op.startswith("s_"):            # a scalar write takes the register's place
                for r in _regs(rest.split(",")[0]):
                    made.pop(r, None)
            continue
        args = [a.strip() for a in re.sub(r"\b(dst_sel|dst_unused|src0_sel|src1_sel|op_sel|row_|quad_|bank_mask|row_mask|bound_ctrl).*", "", rest).split(",")]
        wrote, read = _access(op, args)
        lane = op.startswith(LANE)
        select = _regs(args[-1]) if op.startswith(("v_readlane", "v_writelane")) else set()
        for r in sorted(read | ({"exec"} if lane else set())):
            if r not in made:
                continue
            at, part = made[r]
            if r == "exec":
                need = 4 if lane else 0
            elif r[0] == "v" and r != "vcc":
                need = 1 if part or (lane and not op.startswith("v_writelane")) else 0
            else:
                need = 4 if r in select else 2
            if now - 1 - at < need:
                found.append((kernel, body, r, now - 1 - at, need))
                break
        part = "dst_sel" in rest and "dst_sel:DWORD" not in rest
        for r in wrote:
            made[r] = (now, part)
    return found


def code_object(tmp_path):
    """The gfx950 code object of the built library, and ROCm's tool by name."""
    def tool(t):
        return os.path.join(BIN, t)
    if not os.path.exists(LIB) or not all(shutil.which(tool(t)) for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-objdump", "llvm-readelf")):
        pytest.skip("needs the built library and ROCm's binary tools")
    fat, co = str(tmp_path / "fat.bin"), str(tmp_path / "k.co")
    subprocess.run([tool("llvm-objcopy"), "-O", "binary", "--only-section=.hip_fatbin", LIB, fat], check=True)
    subprocess.run([tool("clang-offload-bundler"), "--type=o", "--unbundle", f"--input={fat}", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950",
                    f"--output={co}"], check=True)
    return co, tool


def test_wait_states(tmp_path):
    co, tool = code_object(tmp_path)
    text = subprocess.run([tool("llvm-objdump"), "-d", "--no-show-raw-insn", co], check=True, capture_output=True, text=True).stdout
    lines = text.splitlines()
    assert any("v_cmpx_lt_u32_sdwa" in x for x in lines)                     # the literal loop is there to be checked
    bad = violations(lines)
    assert not bad, bad[:10]


@pytest.mark.parametrize("code,n", [
    ("v_cmp_gt_u32_e32 vcc, s18, v97\nv_cndmask_b32_e32 v32, 0, v47, vcc", 1),
    ("v_cmp_gt_u32_e32 vcc, s18, v97\ns_nop 0\nv_cndmask_b32_e32 v32, 0, v47, vcc", 1),
    ("v_cmp_gt_u32_e32 vcc, s18, v97\ns_nop 1\nv_cndmask_b32_e32 v32, 0, v47, vcc", 0),
    ("v_cmp_gt_u32_e64 s[4:5], s18, v97\nv_mov_b32_e32 v1, v2\nv_cndmask_b32_e64 v32, 0, v47, s[4:5]", 1),
    ("v_readfirstlane_b32 s5, v1\nv_mov_b32_e32 v2, s5", 1),
    ("v_readfirstlane_b32 s5, v1\ns_mov_b32 s5, 0\nv_mov_b32_e32 v2, s5", 0),
    ("v_cmpx_lt_u32_sdwa vcc, v32, v35 src0_sel:DWORD src1_sel:WORD_1\nv_lshlrev_b64 v[96:97], v32, v[96:97]\ns_nop 1\nv_readfirstlane_b32 s17, v90", 1),
    ("v_cmpx_lt_u32_sdwa vcc, v32, v35 src0_sel:DWORD src1_sel:WORD_1\nv_mov_b32_e32 v1, v2\nv_lshlrev_b64 v[96:97], v32, v[96:97]\ns_nop 1\nv_readfirstlane_b32 s17, v96", 0),
    ("v_lshlrev_b64 v[96:97], v32, v[96:97]\nv_readfirstlane_b32 s17, v96", 1),
    ("v_sub_u32_sdwa v3, v1, v2 clamp dst_sel:BYTE_1 dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_1\nv_min_u32_e32 v3, 8, v3", 1),
    ("v_readlane_b32 s4, v1, s3\ns_nop 2\nv_readlane_b32 s5, v1, s4", 1)])
def test_the_check_finds(code, n):
    assert len(violations(code.splitlines())) == n
