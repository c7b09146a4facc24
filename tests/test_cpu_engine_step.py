"""Host build of the step's continuation and the features' quotients against their plain
formulations (tests/engine_step_check.cpp includes cugo_amd/csrc/engine.h in host code):
the in-place apply with the state put back on failure against probe-then-apply on a copy,
on random games' rows and on rows with random fields changed; the encoder's quotients
against the division, for every value."""

from __future__ import annotations

import os
import shutil
import subprocess
from pathlib import Path

import pytest

REPO = Path(__file__).resolve().parents[1]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_step_continuation_and_quotients_match_plain_formulations(tmp_path):
    if not (Path(HIPCC).exists() or shutil.which("hipcc")):
        pytest.skip("hipcc is not installed")
    exe = tmp_path / "engine_step_check"
    subprocess.run([HIPCC, "-O1", "-std=c++17", "-ffp-contract=off",
                    f"-I{REPO / 'cugo_amd' / 'csrc'}", f"-I{REPO / 'include'}",
                    str(REPO / "tests" / "engine_step_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, timeout=300)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.count("equal") == 2, out.stdout
