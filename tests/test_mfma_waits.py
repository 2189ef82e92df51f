"""The sums of matrix products in the tiles of some ten to a few hundred rows are not read before they are there: the check itself on a
few lines of assembly, and the kernels' assembly as it is built."""
import importlib.util
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _load(name, path):
    spec = importlib.util.spec_from_file_location(name, os.path.join(ROOT, path))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


waits = _load("check_mfma_waits", "tools/check_mfma_waits.py")
ASM = [";;#ASMSTART", "v_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]", ";;#ASMEND"]


@pytest.mark.parametrize("lines,findings", [
    (ASM + ["v_accvgpr_read_b32 v9, a3"], 1),                                        # a copy right behind the product
    (ASM + ["v_accvgpr_read_b32 v9, a3", "s_nop 7", "s_nop 7"], 1),                  # ... in front of the fence
    (ASM + ["s_nop 7", "v_accvgpr_read_b32 v9, a0"], 1),
    (ASM + ["s_nop 7", "s_nop 7", "v_accvgpr_read_b32 v9, a0"], 0),
    (ASM + ["s_waitcnt lgkmcnt(0)", "v_accvgpr_mov_b32 a9, a1"], 1),                 # (a wait for something else is one state)
    (ASM + ASM + ["v_mov_b32 v9, v8"], 0),                                           # the next accumulation is the hardware's matter
    ([".LBB0_1:"] + ASM + ["s_cbranch_scc1 .LBB0_1", "v_accvgpr_read_b32 v9, a0"], 1),
    (["s_branch .LBB0_2", ".LBB0_1:", "v_accvgpr_read_b32 v9, a0", "s_endpgm", ".LBB0_2:"] + ASM + ["s_branch .LBB0_1"], 1),
    (ASM[1:2] + ["v_accvgpr_read_b32 v9, a3"], 0),                                   # (the compiler's own products wait by themselves)
])
def test_the_check(lines, findings):
    assert len(waits.scan(lines)) == findings


@pytest.mark.skipif(not (shutil.which("hipcc") or os.path.exists("/opt/rocm/bin/hipcc")), reason="no compiler")
@pytest.mark.parametrize("src", ["kernels/linear_mid.hip", "hybrid/rows_mid.hip"])
def test_mid_sized_products(src, tmp_path):
    b = _load("repo_build", "build.py")
    path = os.path.join(ROOT, "jax_llama_amd", "csrc", src)
    out = tmp_path / "k.s"
    subprocess.run([b.HIPCC, *b.HIP_FLAGS, *b.FILE_FLAGS.get(os.path.splitext(os.path.basename(src))[0], []), "--cuda-device-only", "-S",
                    path, "-o", str(out)], check=True, capture_output=True)
    text = out.read_text()
    assert text.count("v_mfma") > 100 and not waits.check(text)


def test_the_build_checks_every_source_with_products_in_asm():
    """Also through the headers that it includes."""
    import re
    csrc = os.path.join(ROOT, "jax_llama_amd", "csrc")

    def text_of(path, seen):
        seen.add(path)
        text = open(path).read()
        for name in re.findall(r'#include "([^"]+)"', text):
            at = os.path.normpath(os.path.join(os.path.dirname(path), name))
            if at not in seen and os.path.exists(at):
                text += text_of(at, seen)
        return text

    listed = _load("repo_build", "build.py").ASM_CHECKS
    found = set()
    for part in ("kernels", "hybrid"):
        for name in sorted(os.listdir(os.path.join(csrc, part))):
            if name.endswith(".hip") and re.search(r'asm volatile\([^;]*v_mfma', text_of(os.path.join(csrc, part, name), set())):
                found.add(name[:-4])
    assert found and found <= {src for src, tools in listed.items() if "check_mfma_waits" in tools}
