"""Properties of the built library that its speed depends on."""
import shutil
import subprocess

import pytest


@pytest.mark.skipif(shutil.which("nm") is None, reason="needs nm")
@pytest.mark.parametrize("name", ["rf_denoiser_create", "normal_distribution"])
def test_host_functions_start_on_cache_lines(rf, name):
    """A denoiser's weights are drawn one library call each; a call whose code
    lies across cache lines took 1.7 times as long."""
    from refrakt_amd import build
    out = subprocess.run(["nm", build.LIB], check=True, capture_output=True, text=True).stdout
    at = [int(line.split()[0], 16) for line in out.splitlines() if name in line and line.split()[1] in "TtWw"]
    assert at and all(a % 64 == 0 for a in at), [hex(a) for a in at]
