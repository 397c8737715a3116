"""The pyramid kernels convert their sums under round toward zero. The compiler knows
nothing of the switch, so no other arithmetic may come to lie between it and the switch
back: in the compiled kernels, only the conversions do, and the 0.5 that the octave
step adds before them."""
import os
import re
import shlex
import subprocess

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(REPO, "sift-wgpu_amd")


def test_only_conversions_round_toward_zero(tmp_path):
    obj = "build/kernels_pyramid.o"
    steps = subprocess.run(["make", "-s", "-n", "-B", obj], cwd=PKG, check=True, capture_output=True, text=True).stdout
    cmd = shlex.split(next(x for x in steps.splitlines() if "-c csrc/kernels_pyramid.hip" in x))
    asm = str(tmp_path / "pyramid.s")
    cmd[cmd.index("-c")] = "-S"
    cmd[cmd.index(obj)] = asm
    subprocess.run(cmd + ["--cuda-device-only"], cwd=PKG, check=True, capture_output=True)
    mode, switches = 0, 0
    for line in open(asm):
        op = line.split(";")[0].strip()
        m = re.match(r"s_setreg\S*\s+hwreg\(HW_REG_MODE, 0, 2\), (\S+)", op)
        if m:
            assert int(m.group(1), 0) == (0 if mode else 3), "a switch without its return"
            mode, switches = int(m.group(1), 0), switches + (mode == 0)
        elif mode:
            assert op == "" or re.match(r"s_nop|v_cvt_pk_u8_f32 |v_add_f32(_e32|_e64)? (v\d+), 0\.5, \2$", op), op
    assert mode == 0 and switches > 0
