"""Diagnostics at every supported t length, of a time-domain field (just uploaded)
and of a t-spectral one (after a run), against the oracle's sums of the
downloaded field."""
import numpy as np
import pytest

import oracle_lib as O
from mpc_amd import Propagator, configs, make_inputs

pytestmark = pytest.mark.gpu

# relative to each array's largest value; FP32: the rounding of a transform of that precision
TOL = {"f64": 1e-12, "f32": 1e-5}


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("nx,nt", [(32, 256), (16, 512), (32, 1024), (16, 2048), (16, 4096), (32, 4096)])
def test_diagnostics_at_every_t_length(gpu_lib, prec, nx, nt):
    print(f"case diagnostics nx={nx} nt={nt} prec={prec}", flush=True)
    inp = make_inputs(configs.small(nx, nt))
    with Propagator(inp, prec) as p:
        p.upload(inp.calibrated())
        for domain in ("time", "t-spectral"):
            if domain == "t-spectral":
                p.run(0, 1)
            d, A = p.diagnostics(), p.download()
            dims = O.dims_arr(A.shape)
            ref = {"temp": np.zeros(nt), "spec": np.zeros(nt), "BP1": np.zeros(nx), "BP2": np.zeros(nx)}
            O.oracle().oracle_temp_spec(O.vp(A), O.ip(dims), O.dp(ref["temp"]), O.dp(ref["spec"]))
            O.oracle().oracle_beam_profiles(O.vp(A), O.ip(dims), O.dp(ref["BP1"]), O.dp(ref["BP2"]))
            for n, r in ref.items():
                err = np.abs(d[n] - r).max() / r.max()
                print(f"  {domain} {n}: {err:.2e}", flush=True)
                assert err <= TOL[prec], (domain, n)
            assert abs(d["energy_sum"] - ref["temp"].sum()) <= TOL[prec] * ref["temp"].sum()
