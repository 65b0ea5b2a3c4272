"""The row sweep's branch-free quotients (csrc/sgnx_fastdiv.h) equal IEEE
division bit for bit wherever their range tests let a dividend through."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_branch_free_quotients_equal_ieee_division():
    exe = os.path.join(HERE, "cpp", "sharediv_check")
    if not os.path.exists(exe):
        subprocess.run(["make", "sharediv_check"], cwd=os.path.dirname(exe), check=True)
    out = subprocess.run([exe, "2000000"], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout[-2000:]
