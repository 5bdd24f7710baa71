"""Every address that the kernel for any size and alignment reads along k, walked on the CPU with the kernel's own
functions (csrc/ptl_ragged_piece.hpp): k from one piece to four slabs and one element, every split, both element sizes."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_no_read_outside_of_the_tensor(tmp_path):
    exe = str(tmp_path / "ragged_pieces")
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", os.path.join(ROOT, "pulp-trainlib_amd", "csrc"),
                           os.path.join(ROOT, "tests", "host", "ragged_pieces.cpp"), "-o", exe])
    res = subprocess.run([exe], stdout=subprocess.PIPE, text=True, timeout=300)
    assert res.returncode == 0, res.stdout
