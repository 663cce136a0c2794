"""Wait states in the built null-space kernels: a DPP read or a lane swap needs two
after a VALU write of its source.  The compiler provides them for its own
instructions, not for writes inside asm blocks, so they are counted here in the
assembly of the objects that the build leaves (llvm-objdump)."""
import os
import re
import subprocess

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "radialbasisfinitedifferences.jl_amd")
LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
# 32 lanes a stencil (lane swaps and DPP) and one with 16 (DPP alone)
OBJECTS = ["stencil_ns42_21", "stencil_ns43_21", "stencil_ns57_28", "stencil_nsg42_10", "stencil_nsg47_15",
           "stencil_nsg53_21", "stencil_ns31_15"]
REG = re.compile(r"^[-|]*v\[?(\d+)(?::(\d+))?")


def _regs(arg):
    m = REG.match(arg)
    return range(int(m[1]), int(m[2] or m[1]) + 1) if m else ()


def _hazards(lines):
    """(reads checked, those less than two wait states after a VALU write of their source)"""
    reads, bad, at, written = 0, [], 0, {}  # written: register -> position of its last VALU write
    for line in lines:
        line = line.split("//")[0].strip()
        if not line or line.endswith(":"):
            continue
        op, _, rest = line.partition(" ")
        args = [a.strip() for a in rest.split(",")]
        if op == "s_nop":
            at += int(args[0], 0) + 1
            continue
        swap = op.startswith("v_permlane") and "swap" in op
        if swap or "_dpp" in op or "row_" in rest or "quad_perm" in rest:
            reads += 1
            src = [*_regs(args[0]), *_regs(args[1])] if swap else _regs(args[1])
            if any(at - written.get(r, -9) - 1 < 2 for r in src):
                bad.append(line)
        if op.startswith("v_"):
            for r in [*_regs(args[0]), *(_regs(args[1]) if swap else ())]:
                written[r] = at
        at += 1
    return reads, bad


def test_the_count():
    write, swap = "v_fmac_f64_dpp v[2:3], v[8:9], v[10:11] row_newbcast:3 row_mask:0xf", "v_permlane16_swap_b32_e32 v3, v5"
    dpp = "v_mov_b32_dpp v7, v2 row_shr:1"
    for read in (swap, dpp):
        assert _hazards([write, read])[1] == [read]
        assert _hazards([write, "s_nop 0", read])[1] == [read]
        assert _hazards([write, "s_nop 1", read])[1] == []
        assert _hazards([write, "v_mov_b32 v20, v21", "s_nop 0", read])[1] == []
    assert _hazards([swap, "v_mov_b32_dpp v7, v5 row_shr:1"])[1] != []


@pytest.mark.parametrize("name", OBJECTS)
def test_built_kernels(name, tmp_path):
    obj = os.path.join(PKG, "_build", name + ".o")
    tools = [os.path.join(LLVM, t) for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-objdump")]
    if not os.path.exists(obj) or not all(os.path.exists(t) for t in tools):
        pytest.skip("no built objects or no LLVM tools here")
    fat, code = str(tmp_path / "fat"), str(tmp_path / "code")
    subprocess.run([tools[0], "--dump-section", ".hip_fatbin=" + fat, obj, os.devnull], check=True)
    subprocess.run([tools[1], "--type=o", "--unbundle", "--input=" + fat, "--output=" + code,
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
    p = subprocess.Popen([tools[2], "-d", "--no-show-raw-insn", code], stdout=subprocess.PIPE, text=True)
    reads, bad = _hazards(p.stdout)
    assert p.wait() == 0
    assert reads > 1000 and not bad, bad[:10]
