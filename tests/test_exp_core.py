"""The kernels' own expf on the CPU, every float argument: the header that they are compiled with, and their table."""
import os
import re
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "mako_amd", "csrc")


def test_every_argument():
    src = open(os.path.join(CSRC, "device_math.h")).read()
    table = re.findall(r"0x3f[0-9a-f]{14}", src[src.index("k_exp2_tab"):src.index("};")])
    assert len(table) == 32
    # (the kernels have no other: what they call is the header's, between its bounds)
    assert "return exp_form(__builtin_amdgcn_fmed3f(x, kExpLow, kExpHigh), tab);" in src
    exe, obj = os.path.join(HERE, "cpu", "exp_core_test"), os.path.join(HERE, "cpu", "exp_core_oracle.o")
    flags = ["-O2", "-march=x86-64-v3", "-ffp-contract=off"]
    subprocess.run(["gcc", *flags, "-c", os.path.join(HERE, "..", "oracle", "oracle.c"), "-o", obj], check=True)
    subprocess.run(["g++", *flags, "-std=c++17", "-pthread", os.path.join(HERE, "cpu", "exp_core_test.cpp"), obj, "-o", exe, "-lm"], check=True)
    done = subprocess.run([exe, *table], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout
