"""Row pitches (row_lines in lbm_amd/csrc/layout.h), on the CPU by `layout_check rows`: rows at and next to the lengths
where a line is added keep every property of a layout (elements of their own, alignment, padding that touches nothing
else), and for every length the pitch is the least number of lines or one more where the rule says so."""
import json
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EXE = os.path.join(ROOT, "lbm_amd", "_build", "layout_check")


def test_row_pitches():
    if not os.path.exists(EXE):
        pytest.fail("layout_check not built (python -m lbm_amd.build)")
    p = subprocess.run([EXE, "rows"], capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stdout + p.stderr
    assert json.loads(p.stdout.splitlines()[-1])["rows"] == 3 * 2 * 7 * 3 * 3 * 2 + 4 * 3 * 2 * 4998 * 2
