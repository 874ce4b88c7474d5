"""A read between mflbm_init_phi and the populations on a used handle changes nothing: the phi that
is read, and everything that is set up and run from it, are those of a new handle, bit for bit."""
import pytest

from helpers import assert_same, periodic_drop, small_drainage
from mflbm import gpu

pytestmark = pytest.mark.gpu

CASES = {"drainage": lambda: small_drainage(n=(17, 9, 9), seed=4, radius=2.5, porosity=0.55, jper=1, buffer=2),
         "periodic": lambda: periodic_drop(n=(12, 8, 8), radius=3.0, geo_seed=3)}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("precision", [gpu.FP64, gpu.FP32])
@pytest.mark.parametrize("read", [("phi",), ("c_norm",), ("cn_x", "phi")])
def test_reads_between_phi_and_populations(name, precision, read):
    geo, p = CASES[name]()
    print(f"[gpu-reads] {name} {precision} {read}", flush=True)
    a, b = gpu.Solver(p, geo, precision), gpu.Solver(p, geo, precision)
    a.setup()
    a.run(1, 9)
    for s in (a, b):
        s.init_phi(p["initial_fluid_distribution_option"], p["interface_z0"])
    for field in read:
        a.download(field)
    assert_same(a.download("phi"), b.download("phi"), 0.0, what=f"{name} phi as set")
    for s in (a, b):
        s.init_equilibrium()
        s.color_gradient()
    assert_same(a.download("pdf"), b.download("pdf"), 0.0, what=f"{name} pdf")
    for s in (a, b):
        s.run(1, 20)
    for field in ("pdf", "phi"):
        assert_same(a.download(field), b.download(field), 0.0, what=f"{name} step 20 {field}")


@pytest.mark.parametrize("precision", [gpu.FP64, gpu.FP32])
def test_profile_of_no_steps(precision):
    """no step taken leaves nothing behind: the populations that follow start from the phi as set"""
    geo, p = CASES["drainage"]()
    print(f"[gpu-reads] profile of no steps {precision}", flush=True)
    a, b = gpu.Solver(p, geo, precision), gpu.Solver(p, geo, precision)
    for s in (a, b):
        s.init_phi(p["initial_fluid_distribution_option"], p["interface_z0"])
        if s is a:
            assert s.profile(1, 0)["n_odd"] == 0
        s.init_equilibrium()
    for field in ("pdf", "phi"):
        assert_same(a.download(field), b.download(field), 0.0, what=field)
