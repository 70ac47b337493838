"""The one-launch convolution's plan on the CPU: ``juliavision_amd/csrc/conv_tile_plan.hpp``, which its launch code uses, compiled into
a host program that checks the loads each choice leads to against the tensor's bounds."""
import os
import subprocess
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))


def test_every_weight_load_of_every_choice_is_inside_the_tensor():
    with tempfile.TemporaryDirectory() as tmp:
        exe = os.path.join(tmp, "conv_tile_host_test")
        subprocess.run(["g++", "-O1", "-std=c++17", os.path.join(HERE, "conv_tile_host_test.cpp"), "-o", exe], check=True)
        r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
