"""The words that the one-launch blur reads at an image's edges (csrc/edge_words.h),
all of them, on the CPU: none holds a byte past a row of 4 pixels or more, so that
after a caller's last row nothing of somebody else's is read, and the bytes taken of
them are the clamped pixels."""
import os
import subprocess

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_words_stay_in_the_row(tmp_path):
    exe = str(tmp_path / "edge_words_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror",
                    "-I" + os.path.join(REPO, "sift-wgpu_amd", "csrc"), "-o", exe,
                    os.path.join(REPO, "tests", "c", "edge_words_check.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
    assert r.stdout.strip() == "EDGE_WORDS_OK"
