"""The t-line kernels against the CPU oracle and each other: the exponential of one
step's nonlinear phase (polynomials where a wavefront's phases are all below 1/8 and
losses below 1/32, the general forms above), and reads of a t-spectral field."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle_lib as O
from mpc_amd import Propagator, configs, lib, make_inputs
from mpc_amd._lib import check

pytestmark = pytest.mark.gpu

# field against the oracle, relative L2: the precision forms' bars
TOL = {"f64": 1e-10, "f32": 1e-4}


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("nt", [256, 1024])               # a line within a wavefront, and across two
@pytest.mark.parametrize("phase", [0.01, 0.115, 0.15, 0.6])   # largest per step; every wavefront small, and not
def test_step_exponential_matches_oracle(gpu_lib, prec, nt, phase):
    print(f"case step exponential nt={nt} phase={phase} prec={prec}", flush=True)

    def case(energy):
        inp = make_inputs(configs.small(32, nt, energy=energy, plasm=0, sst_on=1, steps_per_pass=3, passes=2))
        return inp, inp.calibrated()
    inp, A0 = case(1e-6)
    peak = inp.params.gamma2 * (np.abs(A0) ** 2).max() * inp.params.dzz
    inp, A0 = case(1e-6 * phase / peak)
    assert np.isclose(inp.params.gamma2 * (np.abs(A0) ** 2).max() * inp.params.dzz, phase, rtol=1e-9)
    ref, _ = O.run_fixed(inp, A0, 0, 2)
    with Propagator(inp, prec) as p:
        p.upload(A0)
        p.run(0, 2)
        got = p.download()
    err = O.rel_l2(got, ref)
    print(f"  rel_l2={err:.3e}", flush=True)
    assert err <= TOL[prec]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("nx,nt", [(16, 256), (32, 512), (16, 1024), (32, 2048), (16, 4096)])
def test_reads_of_a_spectral_field_agree(gpu_lib, prec, nx, nt):
    """after a run the resident field is t-spectral: download, the float planes
    and the snapshot (which transforms in place) hold the same bits, and none of
    the reads before the snapshot changes what a later run computes"""
    print(f"case reads of a spectral field nx={nx} nt={nt} prec={prec}", flush=True)
    inp = make_inputs(configs.small(nx, nt, steps_per_pass=3, passes=2))
    A0 = inp.calibrated()
    scale = 2.0 ** -3                                      # exact in every format
    with Propagator(inp, prec) as p:
        p.upload(A0)
        p.run(0, 1)
        p.run(1, 1)
        whole = p.download()
    with Propagator(inp, prec) as p:
        p.upload(A0)
        p.run(0, 1)
        first = p.download()
        planes = torch.empty((2, nx, nx, nt), dtype=torch.float32, device="cuda")
        check(lib().mpc_export_planar(p.ctx, C.c_void_p(planes.data_ptr()), scale), "mpc_export_planar")
        p.run(1, 1)
        assert np.array_equal(p.download(), whole)
    with Propagator(inp, prec) as p:
        p.upload(A0)
        p.run(0, 1)
        p.snapshot_begin()
        assert np.array_equal(p.snapshot_wait(), first)
    ref = np.ascontiguousarray(np.moveaxis(first, 0, -1)) * scale      # [t][y][x] to the planes' [y][x][t]
    got = planes.cpu().numpy()
    assert np.array_equal(got[0], ref.real.astype(np.float32))
    assert np.array_equal(got[1], ref.imag.astype(np.float32))
