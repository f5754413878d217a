"""The x/y sweeps' variant of a context that is not tuned: persistent workgroups
only where they measured faster than a workgroup per tile."""
import pytest

from mpc_amd import Propagator, configs, make_inputs

pytestmark = pytest.mark.gpu

PERSISTENT, PER_TILE = 16, 0


@pytest.mark.parametrize("prec,nx,nt,want", [
    # both sides of each line of the rule; at 512 points the persistent form spills and takes twice the time
    ("f32", 64, 256, PER_TILE), ("f32", 128, 256, PERSISTENT), ("f32", 256, 256, PERSISTENT),
    ("f32", 512, 256, PER_TILE),
    ("f64", 64, 512, PER_TILE), ("f64", 128, 512, PERSISTENT), ("f64", 128, 1024, PER_TILE),
    ("f64", 192, 256, PERSISTENT), ("f64", 256, 256, PER_TILE), ("f64", 256, 512, PERSISTENT),
    ("f64", 512, 256, PER_TILE)])
def test_untuned_sweep_variants(gpu_lib, monkeypatch, prec, nx, nt, want):
    print(f"case untuned variants {prec} nx={nx} nt={nt}", flush=True)
    monkeypatch.delenv("MPC_AXIS_VARIANT", raising=False)
    inp = make_inputs(configs.small(nx, nt))
    with Propagator(inp, prec) as p:
        assert p.variants()[1:] == (want, want)
