"""The Jacobi rotation of the pair solves without a GPU: its source on the
host, with reciprocal square roots a unit in the last place off."""
import os
import subprocess

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host")
U = 2.0 ** -53


def test_rotation_is_fp64(tmp_path):
    exe = str(tmp_path / "rotation_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", os.path.join(HERE, "rotation_check.cpp"), "-o",
                    exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300, check=True)
    left, length, tangent = map(float, r.stdout.split())
    # what is left of the element, over r: half a unit each for c^2 - s^2 times
    # apq, for c s d and for their sum (apq, c s d <= r / 2), and one for
    # rounding c and s
    assert left <= 3 * U
    # two rounded squares and products, and c and s themselves
    assert length <= 8 * U
    assert tangent <= 4 * U
