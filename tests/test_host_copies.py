"""The copies' slots without a GPU: the same source on host memory, where
whatever is queued runs as late as the waits allow and the pinned memory lies
between guards."""
import os
import subprocess

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host")
ROOT = os.path.dirname(os.path.dirname(HERE))


def test_every_row_has_its_slot(tmp_path):
    """Rows on both sides of a slot's sizes (256 KB to 4 MB), one of them and
    several: each arrives, and nothing outside the pinned memory is touched."""
    exe = str(tmp_path / "pitched_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", HERE, "-I", os.path.join(ROOT, "include"), "-I",
                    os.path.join(ROOT, "mopac_gpu_amd", "csrc"), os.path.join(HERE, "pitched_check.cpp"), "-o", exe],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
