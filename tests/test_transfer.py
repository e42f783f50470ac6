"""Copies to and from the caller's arrays (lbm_amd/csrc/transfer.cpp), on the CPU: lbm_amd/_build/transfer_check runs
them against a stand-in for the HIP runtime that counts page-locked memory and threads."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EXE = os.path.join(ROOT, "lbm_amd", "_build", "transfer_check")


@pytest.mark.parametrize("case", ["contents", "no_page_locked_memory", "errors", "threads_end", "device_of_the_caller",
                                  "devices_side_by_side", "small_beside_large", "arrays_the_runtime_knows",
                                  "page_locked_by_need"])
def test_transfer(case):
    if not os.path.exists(EXE):
        pytest.fail("transfer_check not built (python -m lbm_amd.build)")
    p = subprocess.run([EXE, case], capture_output=True, text=True, timeout=100)
    assert p.returncode == 0, p.stdout + p.stderr
