"""The inference path's GELU against 64 bits: its polynomial and its FP32 form on
the CPU (tests/cpu/gelu_emul.cpp), and the kernel's on the GPU beside the training
path's."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_gelu_cpu_emulation(tmp_path):
    """the polynomial within 1e-9 of erfc (the bound gelu_poly.h states), the FP32
    form no further from GELU than the erf form over any range of |x|"""
    exe = tmp_path / "gelu_emul"
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", str(exe), os.path.join(ROOT, "tests", "cpu", "gelu_emul.cpp")],
                   check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(out.stdout)
    assert out.returncode == 0 and out.stdout.strip().endswith("OK")


@pytest.mark.gpu
def test_gelu_kernel_accuracy(gpu_lib):
    """a layer whose channel map is the identity and whose mode rows are zero
    leaves GELU of its input: without and with the pre-activations kept the
    inference and the training form.  In |x| / 2, over each range and sign, the
    inference form's rms error is no larger than the training form's (1% for the
    sampling of the two)"""
    from scipy.special import erfc

    from mpc_amd.fno import DArr, Ops
    W, T, n2, npos = 8, 256, 2, 256
    rng = np.random.default_rng(2)
    edges = [0, 0.01, 0.1, 0.5, 1, 2, 4, 8, 16]
    o = Ops()
    v = np.empty((W, npos, T), dtype=np.float32)
    for c in range(W):                                    # a channel per range, both signs
        v[c] = rng.uniform(edges[c], edges[c + 1], (npos, T)) * rng.choice([-1, 1], (npos, T))
    eye, zero = DArr.of(np.eye(W)), DArr.of(np.zeros(W))
    V6, C1 = DArr((W, npos, n2)).fill(0.0), DArr((W, npos, n2))
    Gt, Ft = o.pack(DArr((n2, T)).fill(0.0), 2, n2, T), o.pack(DArr((T, n2)).fill(0.0), 3, T, n2)
    err = {}
    for form in ("inference", "training"):
        out = DArr(v.shape)
        o.column(1, W, npos, T, n2, DArr.of(v), W * npos * T, eye, zero, V6=V6, Gt=Gt, Ft=Ft, act=True, out=out, C1=C1,
                 zs=DArr(v.shape) if form == "training" else None)
        x = v.astype(np.float64)
        err[form] = np.abs(out.numpy() - 0.5 * x * erfc(-x / np.sqrt(2))) / (0.5 * np.abs(x))
    for c in range(W):
        for sg in (-1, 1):
            at = np.sign(v[c]) == sg
            a, b = (np.sqrt(np.mean(err[f][c][at] ** 2)) for f in ("inference", "training"))
            m = [err[f][c][at].max() for f in ("inference", "training")]
            print(f"case gelu {'-+'[sg > 0]}|x| {edges[c]}-{edges[c + 1]}: rms {a:.2e} (training {b:.2e}), "
                  f"max {m[0]:.2e} ({m[1]:.2e})", flush=True)
            assert a <= 1.01 * b
