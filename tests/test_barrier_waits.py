"""attn_packed_kernel fills a buffer in LDS behind a bare s_barrier: what a wave asked for before it - its share of the next chunk, its reads of the
one before - has to be waited for in front of it, in every copy the compiler makes of the loop.  Read off the compiler's own assembly."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="no hipcc")
def test_barriers_stand_behind_both_waits(tmp_path):
    src = tmp_path / "kernels.hip"
    src.write_text('#include "attn_packed.h"\n' + "".join(
        f"template __global__ void jitnn::attn_packed_kernel<{d}>(const float *, const _Float16 *, float *, int, int, int, int, int, float);\n" for d in (64, 128)))
    flags = re.search(r"^FLAGS = (.*?[^\\])\n", (ROOT / "jitnn_amd/csrc/Makefile").read_text(), re.M | re.S).group(1).replace("\\\n", " ").replace("$(ARCH)", "gfx950")
    asm = tmp_path / "kernels.s"
    subprocess.run([HIPCC, *flags.split(), "-I", str(ROOT / "jitnn_amd/csrc"), "--cuda-device-only", "-S", "-o", str(asm), str(src)], check=True, capture_output=True)
    lines = [line.strip() for line in asm.read_text().splitlines()]
    code = [line for line in lines if line and not line.startswith((";", "."))]
    at = [i for i, line in enumerate(code) if line.startswith("s_barrier")]
    assert len(at) == 4  # two loops, with and without the mask, for each head size
    for i in at:
        assert re.fullmatch(r"s_waitcnt vmcnt\(0\) lgkmcnt\(0\)", code[i - 1]), code[i - 1]
