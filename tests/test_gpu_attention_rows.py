"""The attention of long prompts by itself (tests/attention_rows_test.hip, built with the library): the rounding of the weights, and
rows of one wave that rescale their outputs in different chunks, with one and two tiles of rows per wave, against FP64."""
import subprocess
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu

ROOT = Path(__file__).resolve().parent.parent
PROGRAM = ROOT / "tests" / "build" / "attention_rows_test"


def test_attention_rows():
    if not PROGRAM.exists():
        subprocess.run(["make", "-C", str(ROOT / "jitnn_amd" / "csrc"), "tests"], check=True)
    done = subprocess.run([str(PROGRAM)], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0 and done.stdout.endswith("all hold\n"), done.stdout + done.stderr
