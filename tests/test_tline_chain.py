"""The t-line transform with cached twiddle powers, as persistent workgroups run
it, emulated on the CPU (tests/cpu/tline_chain_emul.cpp) at every supported t
length, both directions and precisions: the bits of the form that reads the
twiddle table."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_tline_cached_twiddles_cpu_emulation(tmp_path):
    exe = tmp_path / "tline_chain_emul"
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", str(exe),
                    os.path.join(ROOT, "tests", "cpu", "tline_chain_emul.cpp")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    print(out.stdout)
    assert out.returncode == 0 and out.stdout.strip().endswith("OK")
