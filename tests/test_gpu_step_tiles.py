"""GPU parity of the step at the geometries where its boxes can go wrong (boxes with no node to
compute, boxes without solid, a single box, rows just past a box edge) and where its one
boundary launch can (open boundaries of every kind on a periodic y axis, whose copies share
cells with them, down to four planes).  FP64, so the state must equal the oracle's bit for
bit."""
import numpy as np
import pytest

import oracle as O
from helpers import assert_same, periodic_drop, small_drainage
from mflbm import gpu

pytestmark = pytest.mark.gpu


def solid_block(n, seed, jper=1):
    """a sphere pack whose middle third along z and lower half along y are solid, except for one
    channel that keeps the ends connected"""
    geo, p = small_drainage(n=n, seed=seed, radius=3.0, porosity=0.6, jper=jper, buffer=2)
    nz, ny, nx = geo.shape
    geo[nz // 3:2 * nz // 3] = 1
    geo[2:-2, :ny // 2] = 1
    geo[2:-2, ny // 2 + 1:ny // 2 + 4, nx // 2:nx // 2 + 3] = 0
    return geo, p


def no_solid(n, seed):
    geo, p = small_drainage(n=n, seed=seed, radius=3.0, porosity=0.95, jper=1, buffer=2)
    return np.zeros_like(geo), p


CASES = {
    "solid_boxes": lambda: solid_block((40, 36, 33), 3),
    "solid_boxes_ywalls": lambda: solid_block((35, 33, 30), 4, jper=0),
    "no_solid": lambda: no_solid((18, 17, 13), 5),
    "one_box": lambda: small_drainage(n=(12, 8, 5), seed=2, radius=2.0, porosity=0.6, jper=1, buffer=1),
    "velocity_in_convective_out_yper": lambda: small_drainage(n=(11, 9, 14), seed=6, radius=2.5, porosity=0.55, jper=1,
                                                              buffer=2, inlet=1, outlet=1),
    "four_planes_convective_yper": lambda: small_drainage(n=(10, 6, 4), seed=2, radius=1.5, porosity=0.7, jper=1,
                                                          buffer=1, inlet=1, outlet=1),
    "four_planes_zouhe_yper": lambda: small_drainage(n=(9, 5, 4), seed=3, radius=1.5, porosity=0.7, jper=1, buffer=1),
    # periodic axes of 8 nodes, the fewest whose ghost phi the collision writes, and of 7
    "periodic_8_8": lambda: periodic_drop(n=(12, 8, 8), radius=3.0, geo_seed=3),
    "periodic_7_8": lambda: periodic_drop(n=(12, 7, 8), radius=3.0, geo_seed=4),
    "periodic_8_7": lambda: periodic_drop(n=(12, 8, 7), radius=3.0, geo_seed=5),
    "one_past_a_box": lambda: small_drainage(n=(17, 9, 9), seed=4, radius=2.5, porosity=0.55, jper=1, buffer=2),
}


@pytest.mark.parametrize("name", list(CASES))
def test_steps_bitwise(name):
    geo, p = CASES[name]()
    print(f"[gpu-step-tiles] {name} {geo.shape}", flush=True)
    o, g = O.Oracle(p, geo), gpu.Solver(p, geo, gpu.FP64)
    assert g.gradient_path() == "tiles"
    o.setup()
    g.setup()
    for t in range(1, 4):
        o.step(t)
        g.step(t)
        for field in ("pdf", "phi", "cn_x", "cn_y", "cn_z", "c_norm"):
            assert_same(g.download(field), o.array(field), 0.0, what=f"{name} step {t} {field}")
    o.run(4, 30)
    g.run(4, 30)
    for field in ("pdf", "phi") + (("convec",) if p["outlet_bc"] == 1 else ()):
        assert_same(g.download(field), o.array(field), 0.0, what=f"{name} step 33 {field}")


@pytest.mark.parametrize("n", [(11, 7, 6), (12, 8, 9), (13, 17, 8), (25, 9, 13)])
def test_fp32_boxes_match_the_split_chain(n):
    """FP32 at the edges of its 12 x 8 x 4 and 16 x 8 x 4 boxes, against the kernels of one stage
    each.  Contraction is allowed in FP32, so the two round differently; the bound is that of the
    parity test of the two paths."""
    geo, p = small_drainage(n=n, seed=7, radius=2.0, porosity=0.6, jper=1, buffer=1)
    print(f"[gpu-step-tiles] fp32 {n}", flush=True)
    a, b = gpu.Solver(p, geo, gpu.FP32), gpu.Solver(p, geo, gpu.FP32, split_gradient=True)
    for s in (a, b):
        s.setup()
        s.run(1, 30)
    for field in ("pdf", "phi"):
        assert_same(a.download(field), b.download(field), 1e-5, what=f"{n} {field}")


def test_phi_read_first_leaves_the_normals_to_bring_up():
    """a read of phi brings up phi alone; a read of the normals after it still matches the oracle"""
    geo, p = CASES["one_past_a_box"]()
    o, g = O.Oracle(p, geo), gpu.Solver(p, geo, gpu.FP64)
    print("[gpu-step-tiles] phi before normals", flush=True)
    for s in (o, g):
        s.setup()
        s.run(1, 7)
    for field in ("phi", "cn_x", "phi", "c_norm", "cn_z"):
        assert_same(g.download(field), o.array(field), 0.0, what=field)
    o.run(8, 5)
    g.run(8, 5)
    for field in ("phi", "pdf"):
        assert_same(g.download(field), o.array(field), 0.0, what=field)


@pytest.mark.parametrize("name", ["one_past_a_box", "periodic_8_8", "velocity_in_convective_out_yper"])
def test_populations_started_anew_from_the_phi_of_a_run(name):
    """the boxes leave most solid nodes' phi behind; populations initialised from it after a run are
    those of the kernels of one stage each, which write it in every step"""
    geo, p = CASES[name]()
    print(f"[gpu-step-tiles] init after a run {name}", flush=True)
    a, b = gpu.Solver(p, geo, gpu.FP64), gpu.Solver(p, geo, gpu.FP64, split_gradient=True)
    for s in (a, b):
        s.setup()
        s.run(1, 9)
        s.init_equilibrium()
    inside = (..., slice(1, -1), slice(1, -1), slice(1, -1))
    assert_same(a.download("pdf")[inside], b.download("pdf")[inside], 0.0, what=f"{name} pdf")


@pytest.mark.parametrize("n, precision", [((49, 41, 45), gpu.FP64), ((50, 39, 46), gpu.FP32), ((33, 41, 44), gpu.FP64),
                                          ((37, 33, 41), gpu.FP32)])
def test_domains_around_the_change_of_box_and_workgroup_sizes(n, precision):
    """the last sizes with small boxes and with one-wave collide workgroups and the first beyond them:
    FP64 against the oracle, FP32 against the kernels of one stage each (as above)"""
    geo, p = small_drainage(n=n, seed=9, radius=3.5, porosity=0.55, jper=1, buffer=2)
    print(f"[gpu-step-tiles] sizes {n} {precision}", flush=True)
    g = gpu.Solver(p, geo, precision)
    o = O.Oracle(p, geo) if precision == gpu.FP64 else gpu.Solver(p, geo, precision, split_gradient=True)
    for s in (o, g):
        s.setup()
        s.run(1, 30)
    for field in ("pdf", "phi"):
        if precision == gpu.FP64:
            assert_same(g.download(field), o.array(field), 0.0, what=f"{n} {field}")
        else:
            assert_same(g.download(field), o.download(field), 1e-5, what=f"{n} {field}")


@pytest.mark.parametrize("name", ["one_past_a_box", "periodic_8_8"])
@pytest.mark.parametrize("precision", [gpu.FP64, gpu.FP32])
def test_a_second_start_on_a_handle_is_the_first(name, precision):
    """populations and phi set up again after a run are those of a new handle, bit for bit: the phi of
    solid nodes is the one that init_phi sets, not the last step's"""
    geo, p = CASES[name]()
    print(f"[gpu-step-tiles] second start {name} {precision}", flush=True)
    a, b = gpu.Solver(p, geo, precision), gpu.Solver(p, geo, precision)
    a.setup()
    a.run(1, 9)
    for s in (a, b):
        s.setup()
    for field in ("pdf", "phi"):
        assert_same(a.download(field), b.download(field), 0.0, what=f"{name} {field}")
    for s in (a, b):
        s.run(1, 30)
    for field in ("pdf", "phi"):
        assert_same(a.download(field), b.download(field), 0.0, what=f"{name} step 30 {field}")
