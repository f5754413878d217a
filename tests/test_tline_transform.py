"""The t-line transform's step across wavefronts and its frequency order,
emulated on the CPU thread by thread (tests/cpu/tline_emul.cpp) at every
supported t length, both directions and precisions, against a brute-force
DFT: 1e-14 (FP64) and 2e-6 (FP32), the bounds of the stage emulation."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_tline_transform_cpu_emulation(tmp_path):
    exe = tmp_path / "tline_emul"
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", str(exe), os.path.join(ROOT, "tests", "cpu", "tline_emul.cpp")],
                   check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    print(out.stdout)
    assert out.returncode == 0 and out.stdout.strip().endswith("OK")
