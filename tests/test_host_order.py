"""The host core's reordered and scaled matrix (host_order.cpp), entry for entry and bit for bit."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_matrix_in_a_given_order(tmp_path):
    exe = str(tmp_path / "host_order")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(HERE, "..", "include"), os.path.join(HERE, "host_order.cpp"),
                    "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
