"""Device-to-host copies (rf_stage.cpp) on a fake runtime of two devices, on
the CPU: what one GPU cannot show."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def stage(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("stage") / "stage")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(HERE, "fake_hip"),
                    os.path.join(HERE, "stage_driver.cpp"), "-o", exe], check=True)
    return lambda which: subprocess.run([exe, which], capture_output=True, text=True, timeout=60)


def test_copies_on_another_devices_stream(stage):
    """A context of one device, a thread whose current device is another: copies
    of every length work and leave the current device alone."""
    r = stage("other_device")
    assert r.returncode == 0, r.stdout


def test_copies_while_staging_fails(stage):
    """An event that cannot be recorded, at once or after some transfers: the
    bytes arrive by the plain copy, and the next copy is staged again."""
    r = stage("failing_stage")
    assert r.returncode == 0, r.stdout


@pytest.mark.parametrize("kind", ["pinned", "device", "managed", "unregistered"])
def test_destinations_the_runtime_knows(stage, kind):
    """Pinned, device and managed memory take one transfer; only memory that the
    runtime does not know is written by the host's threads."""
    r = stage(kind)
    assert r.returncode == 0, r.stdout


def test_more_threads_than_stages(stage):
    """Pinned memory and threads stay those of two stages; the other copies are
    plain ones instead of waiting for a stage made for them."""
    r = stage("many_threads")
    assert r.returncode == 0, r.stdout
