"""Runs the device check of the products, folds and joins that the kernels stand on
(tests/native/gl64_folds_check.hip, built by triton-vm-prover_amd/Makefile): the
borrow or carry they set aside, which random operands take once in 2^32, in most of
the operands, in each width and with each form of mask the kernels use."""
import os
import subprocess

import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

BIN = os.path.join(ROOT, "triton-vm-prover_amd", "_build", "gl64_folds_check")


def test_gl64_rare_folds_match_u128():
    assert os.path.exists(BIN), "gl64_folds_check not built (run __graft_entry__.build())"
    r = subprocess.run([BIN], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "folds bad=0" in r.stdout
