"""The t-line kernel's exponential of one step's nonlinear phase against the
CPU oracle: polynomials where a wavefront's phases are all below 1/8 (and
losses below 1/32), the general forms above it."""
import numpy as np
import pytest

import oracle_lib as O
from mpc_amd import Propagator, configs, make_inputs

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
