"""The row and table indices of the cropped, corrected image store, checked on the host over
all image sizes of a few padded ones, odd and even (tests/cpp/crop_rows.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_crop_rows(tmp_path):
    exe = str(tmp_path / "crop_rows")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "fastimaging_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "crop_rows.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
