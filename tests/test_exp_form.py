"""The kernels' form of expf on the CPU, every float argument (the device itself: test_gpu_parity.py)."""
import os
import re
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_every_argument():
    src = open(os.path.join(HERE, "..", "mako_amd", "csrc", "device_math.h")).read()
    table = re.findall(r"0x3f[0-9a-f]{14}", src[src.index("k_exp2_tab"):src.index("};")])
    assert len(table) == 32
    exe = os.path.join(HERE, "cpu", "exp_form")
    subprocess.run(["gcc", "-O2", "-march=x86-64-v3", "-ffp-contract=off", "-pthread", os.path.join(HERE, "cpu", "exp_form.c"),
                    os.path.join(HERE, "..", "oracle", "oracle.c"), "-o", exe, "-lm"], check=True)
    done = subprocess.run([exe, *table], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout
