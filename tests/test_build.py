"""The host code of the extension compiles without a warning."""
import os
import shutil
import subprocess

import pytest

from daisy_amd import build


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include"), reason="needs the host compiler and ROCm's headers")
def test_the_extension_compiles_without_warnings():
    cmd = build._native_command()
    assert "-w" not in cmd and {"-Wall", "-Wextra"} <= set(cmd)
    r = subprocess.run([*cmd, "-Werror", "-fsyntax-only", build.NATIVE_SOURCE], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-4000:]
