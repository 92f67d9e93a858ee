"""The weight-only 128-row kernel and the persistent tile kernel issue their MFMAs through inline assembly, so the compiler does not keep the wait states of a
matrix instruction around them: the source does, as long as the register allocator leaves the accumulators where they are.
This reads the code objects that the build here made and checks every one of them (no GPU)."""
import os
import re
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OBJ = os.path.join(REPO, "ms_custom_ops_amd", "lib", "obj", "gmm_rows_a16w8.o")
LLVM = "/opt/rocm/llvm/bin"
BEFORE, BEHIND = 2, 12   # states without a vector write of an operand in front, without an access to the result behind
MFMAS = ("v_mfma_f32_16x16x32", "v_mfma_i32_16x16x64")


def _regs(operands):
    found = set()   # (accumulation registers: from 1000 on)
    for bank, a, lo, hi in re.findall(r"\b([va])(?:(\d+)|\[(\d+):(\d+)\])", operands):
        first = 1000 * (bank == "a")
        found |= {first + int(a)} if a else set(range(first + int(lo), first + int(hi) + 1))
    return found


def _violations(lines):
    """lines: (mnemonic, operand text) in order.  Every MFMA that breaks a rule, as text."""
    near = set()   # (only what stands around an MFMA is looked at)
    for i, (name, _) in enumerate(lines):
        if name.startswith(MFMAS):
            near.update(range(max(0, i - BEFORE), min(len(lines), i + BEHIND + 1)))
    ins = [(name, [_regs(o) for o in ops.split(",")] if ops and i in near else [], ops) for i, (name, ops) in enumerate(lines)]
    states = [int(ops) + 1 if name == "s_nop" else 1 for name, _, ops in ins]
    bad = []
    for i, (name, ops, text) in enumerate(ins):
        if not name.startswith(MFMAS):
            continue
        result, a, b, c = ops[:4]
        if result != c and text.split(",")[3].strip() != "0":   # (a tile's first products replace the accumulators)
            bad.append("moved accumulator: " + text)
        j, seen = i - 1, 0
        while j >= 0 and seen < BEFORE:
            if ins[j][0].startswith("v_") and "mfma" not in ins[j][0]:
                written = ins[j][1][0] | (ins[j][1][1] if "swap" in ins[j][0] else set())
                if written & (a | b):
                    bad.append("%s %s in front of %s" % (ins[j][0], ins[j][2], text))
            seen += states[j]
            j -= 1
        j, seen = i + 1, 0
        while j < len(ins) and seen < BEHIND and ins[j][0] != "s_endpgm":
            mfma = "mfma" in ins[j][0]
            touched = ins[j][1][1] | ins[j][1][2] if mfma else set().union(set(), *ins[j][1])   # (the next sum into the same registers is in order)
            if touched & result:
                bad.append("%s %s behind %s" % (ins[j][0], ins[j][2], text))
            seen += states[j]
            j += 1
    return bad


def test_the_rules_find_what_they_are_for():
    mfma = ("v_mfma_f32_16x16x32_bf16", " v[0:3], v[4:7], v[8:11], v[0:3]")
    assert not _violations([("v_mov_b32", " v4, v20"), ("s_nop", "1"), mfma, ("s_nop", "11"), ("v_add_f32", " v20, v0, v1")])
    assert _violations([("v_mov_b32", " v4, v20"), ("s_nop", "0"), mfma])
    assert _violations([mfma, ("s_nop", "10"), ("v_add_f32", " v20, v0, v1")])
    assert _violations([("v_mfma_f32_16x16x32_bf16", " v[0:3], v[4:7], v[8:11], v[12:15]")])
    first = ("v_mfma_i32_16x16x64_i8", " a[0:3], v[4:7], v[8:11], 0")
    assert not _violations([("v_accvgpr_read_b32", " v4, a0"), ("s_nop", "1"), first, ("v_add_u32", " v0, v1, v2"), ("s_nop", "10"), ("v_accvgpr_read_b32", " v20, a3")])
    assert _violations([first, ("s_nop", "10"), ("v_accvgpr_read_b32", " v20, a3")])
    assert _violations([("v_accvgpr_read_b32", " v4, a9"), first])
    assert _violations([("v_mfma_i32_16x16x64_i8", " a[0:3], v[4:7], v[8:11], a[4:7]")])


def test_inline_mfmas_keep_their_wait_states(tmp_path):
    if not os.path.exists(OBJ) or not os.path.exists(os.path.join(LLVM, "llvm-objdump")):
        pytest.skip("needs the object files of an in-tree build and the ROCm binary tools")
    fat, code = str(tmp_path / "fat"), str(tmp_path / "code")
    subprocess.check_call([os.path.join(LLVM, "llvm-objcopy"), "--dump-section", ".hip_fatbin=" + fat, OBJ, str(tmp_path / "copy.o")])
    subprocess.check_call([os.path.join(LLVM, "clang-offload-bundler"), "--unbundle", "--type=o", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", "--input=" + fat,
                           "--output=" + code])
    text = subprocess.run([os.path.join(LLVM, "llvm-objdump"), "-d", code], check=True, capture_output=True, text=True).stdout
    assert "scratch_" not in text
    seen = 0
    for kernel in re.split(r"^[0-9a-f]+ <", text, flags=re.M)[1:]:
        lines = [(m[1], m[2].split("//")[0].strip()) for m in re.finditer(r"^\t(\S+)(.*)$", kernel, flags=re.M)]
        seen += sum(name.startswith("v_mfma") for name, _ in lines)
        assert _violations(lines) == [], kernel[:80]
    assert seen >= 1000


@pytest.mark.parametrize("unit", ["%s%s" % (layout, out) for layout in ("packed", "nk", "kn") for out in ("", "_bf16", "_f16", "_bf16_silu", "_f16_silu")])
def test_the_persistent_tile_kernel_keeps_them_too(unit, tmp_path, monkeypatch):
    monkeypatch.setitem(globals(), "OBJ", os.path.join(os.path.dirname(OBJ), "gmm_tile4m_%s.o" % unit))
    test_inline_mfmas_keep_their_wait_states(tmp_path)


@pytest.mark.parametrize("unit", ["a16w8_bf16_kn", "a16w8_f16_packed", "a16w8_f16_kn", "a16w4_bf16", "a16w4_f16"])
def test_the_other_types_and_layouts_keep_them_too(unit, tmp_path, monkeypatch):
    monkeypatch.setitem(globals(), "OBJ", OBJ.replace("a16w8.o", unit + ".o"))
    test_inline_mfmas_keep_their_wait_states(tmp_path)
