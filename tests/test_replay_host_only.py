"""The sanitizer build of the C replay makes no device call where a GPU may be (one run
of it there did not end): with a GPU's device node present it stops after the host
checks, also where the checks of tests/test_sanitizers.py start it."""
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(REPO, "sift-wgpu_amd")


def _replay(tmp_path, node, *flags):
    exe = str(tmp_path / "replay")
    subprocess.run(["gcc", "-O1", "-std=c11", "-D_DEFAULT_SOURCE", "-DREPLAY_GPU_NODE=\"%s\"" % node, *flags,
                    "-I" + os.path.join(REPO, "include"), os.path.join(REPO, "tests", "c", "arm_replay.c"),
                    "-o", exe, "-L" + PKG, "-lsift_hip", "-lm", "-Wl,-rpath," + PKG], check=True)
    # (no leak check: the HIP runtime that the library links keeps what it allocates)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0")
    env.pop("SIFT_REPLAY_DEVICE", None)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60, env=env)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout.splitlines()


def test_sanitized_replay_stops_after_the_host_checks(tmp_path):
    assert _replay(tmp_path, "/dev/null", "-fsanitize=address") == ["host checks only", "ARM_REPLAY_NO_DEVICE"]


@pytest.mark.skipif(os.path.exists("/dev/kfd"), reason="makes the calls that reach a device")
def test_without_a_gpu_the_calls_are_made(tmp_path):
    assert _replay(tmp_path, str(tmp_path / "none"), "-fsanitize=address") == ["ARM_REPLAY_NO_DEVICE"]
    assert _replay(tmp_path, "/dev/null") == ["ARM_REPLAY_NO_DEVICE"]
