"""FP64 quotients by a shared divisor (flowvc-1_amd/csrc/fvc_div.h, the
Cartesian kernels' cells, time locations and RK4 sixths) against the division,
bit for bit."""
import os
import subprocess

import cases


def test_div_near_is_the_division(tmp_path):
    exe = os.path.join(str(tmp_path), "div_check")
    src = os.path.join(cases.REPO, "tests", "native", "div_check.c")
    inc = os.path.join(cases.REPO, "flowvc-1_amd", "csrc")
    subprocess.run(["gcc", "-O2", "-std=c11", "-mfma", "-ffp-contract=off", "-I" + inc, src, "-o", exe, "-lm"], check=True)
    out = subprocess.run([exe, "200000"], capture_output=True, text=True, check=True).stdout.splitlines()
    n, bad, ranged = (int(w) for w in out[-1].split())
    assert n == 96 * 200000 and ranged == 1
    assert bad == 0, out[:10]
