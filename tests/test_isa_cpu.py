"""Checks of the gfx950 assembly that the compiler makes of the library's sources (no GPU needed)."""
import importlib.util
import os
import re
import subprocess

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "amdgpu.jl_amd")


def _assembly(source, out):
    spec = importlib.util.spec_from_file_location("_rk_build_flags", os.path.join(PKG, "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    flags = [f for f in build.FLAGS if not f.startswith("-Rpass")]
    subprocess.run([build.HIPCC, *flags, "--cuda-device-only", "-S", os.path.join(PKG, "csrc", source), "-o", str(out)], check=True, capture_output=True)
    return out.read_text().splitlines()


def _scalar_registers(text):
    regs = set()
    for lo, hi, one in re.findall(r"\bs(?:\[(\d+):(\d+)\]|(\d+)\b)", text):
        regs |= {int(one)} if one else set(range(int(lo), int(hi) + 1))
    return regs


def _early_reads(lines):
    """Vector compares inside asm statements, and those of them whose scalar result a vector instruction reads with fewer
    than two wait states in between (an instruction is one, s_nop N is N + 1)."""
    code, inside = [], False
    for l in lines:
        inside = "#ASMSTART" in l or (inside and "#ASMEND" not in l)
        l = l.split(";")[0].strip()
        if re.match(r"[vs]_|global_|ds_|buffer_|flat_|scratch_", l):
            code.append((l, inside))
    compares, early = 0, []
    for i, (l, asm) in enumerate(code):
        if not asm or not l.startswith("v_cmp"):
            continue
        compares += 1
        written, states = _scalar_registers(l.split(",")[0].split(None, 1)[1]), 0
        for k, _ in code[i + 1:]:
            if states >= 2:
                break
            if k.startswith("v_") and "," in k and _scalar_registers(k.split(",", 1)[1]) & written:
                early.append((l, k))
                break
            states += int(k.split()[1], 0) + 1 if k.startswith("s_nop") else 1
    return compares, early


def test_early_reads_are_seen():
    asm = [";;#ASMSTART", "v_cmp_ne_u32_e64 s[0:1], 0, v3", ";;#ASMEND"]
    use = ["v_bitop3_b32 v4, -1, s1, v3 bitop3:0x90"]
    for between, bad in (([], 1), (["s_nop 0"], 1), (["v_bfe_i32 v5, v2, 1, 1"], 1), (["s_nop 1"], 0), (["s_nop 0", "v_bfe_i32 v5, v2, 1, 1"], 0)):
        compares, early = _early_reads(asm + between + use)
        assert compares == 1 and len(early) == bad
    assert _early_reads(asm + ["v_mov_b32_e32 v1, s2"] + use)[1] != [] and _early_reads(["v_cmp_ne_u32_e64 s[0:1], 0, v3"] + use) == (0, [])


@pytest.mark.timeout(300)
def test_masks_of_asm_compares_are_read_late_enough(tmp_path):
    """The digit match of the sorts writes lane masks with compares in an asm statement; the compiler does not keep the two
    wait states a vector instruction needs before it may read them, so the statement has to."""
    compares, early = _early_reads(_assembly("rk_sort.hip", tmp_path / "rk_sort.s"))
    assert compares >= 8 * 24                # six key types, sort and sortperm, small and large sorts
    assert not early, f"{len(early)} of {compares}: {early[0]}"
