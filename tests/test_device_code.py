"""CPU checks of the AMD assembly that this tree's HIP sources compile to."""
import os
import re
import shutil
import subprocess

import pytest

from conftest import ROOT

PKG = os.path.join(ROOT, "moe-680m_amd")


def kernels(asm):
    """{symbol: body} of the kernels and device functions of an assembly file."""
    return dict(re.findall(r"^(_Z\w+):[^\n]*\n(.*?)^\.Lfunc_end", asm, re.S | re.M))


def inline_valu(body):
    """Vector instructions written in inline asm (an empty asm statement or a wait is none)."""
    blocks = re.findall(r";;#ASMSTART\n(.*?);;#ASMEND", body, re.S)
    return [i.strip() for b in blocks for i in b.splitlines() if re.match(r"\s*v_", i)]


@pytest.mark.parametrize("name", ["k_route", "k_prefill"])
def test_no_inline_asm_valu_beside_mfma(name, tmp_path):
    """The compiler puts the wait states that an MFMA's result and operand registers need in
    front of every later vector instruction -- except those in inline asm, which it does not
    look into.  So no kernel with MFMAs may hold one."""
    if not shutil.which("make") or not os.path.exists("/opt/rocm/bin/hipcc"):
        pytest.fail("hipcc is needed to compile the sources")
    out = tmp_path / f"{name}.s"
    r = subprocess.run(["make", "-C", PKG, f"ASM_DIR={tmp_path}", str(out)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    mfma = {k: b for k, b in kernels(out.read_text()).items() if "v_mfma_" in b}
    assert len(mfma) >= 16, sorted(mfma)  # 18 router products; 8 gate/up and 8 down kernels
    bad = {k: inline_valu(b)[:1] for k, b in mfma.items() if inline_valu(b)}
    assert not bad, bad
