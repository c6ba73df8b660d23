"""A libcowsdm.so of another version, or older than the package within a
version, is refused with a message that says so."""

from __future__ import annotations

import os
import subprocess
import sys
from pathlib import Path

import pytest

from copy_on_write_sdm_amd import _native as nat


@pytest.mark.parametrize("version,message", [
    (nat.ABI_VERSION - 1, "ABI version mismatch"),
    (nat.ABI_VERSION, "older than this package, build it again")])
def test_other_builds_are_refused(tmp_path, version, message):
    library = tmp_path / "libcowsdm.so"
    source = tmp_path / "version.c"
    source.write_text(f"int cowsdm_abi_version(void) {{ return {version}; }}\n")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(library), str(source)], check=True)
    run = subprocess.run(
        [sys.executable, "-c", "from copy_on_write_sdm_amd import _native; _native.lib()"],
        env={**os.environ, "COWSDM_LIBRARY": str(library)}, text=True, capture_output=True,
        cwd=Path(__file__).resolve().parent.parent)
    assert run.returncode != 0
    assert f"RuntimeError: {library}" in run.stderr or "RuntimeError: libcowsdm.so" in run.stderr
    assert message in run.stderr
