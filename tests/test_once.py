"""Constant buffers made on first use (rf_once.hpp), on the CPU."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_a_buffer_that_could_not_be_filled_is_not_kept(tmp_path):
    """The density estimation's chord table bounds its loops over columns: after
    a failed fill it is made again, never read as it was allocated."""
    exe = str(tmp_path / "once")
    subprocess.run(["g++", "-std=c++17", os.path.join(HERE, "once_driver.cpp"), "-o", exe], check=True)
    assert subprocess.run([exe]).returncode == 0
