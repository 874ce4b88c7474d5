"""Small ensembles run a wave per workgroup, large ones four: a domain's result is the same bits
alone (small) and among others that stop at other checks (large)."""
import numpy as np
import pytest

from mflbm import cases, config, ensemble

pytestmark = pytest.mark.gpu


def test_a_domain_alone_and_in_a_large_ensemble():
    nx, ny, nz = 20, 16, 24
    p = config.derive(cases.periodic_control(n=(nx, ny, nz), body_force=1e-6, option=1, interface_z0=float(nz + 10)))
    geos = np.stack([cases.geometry.sphere_pack((nz, ny, nx), 3.0, 0.6, s, periodic=(True, True, False))
                     for s in range(4, 28)])
    many = ensemble.Ensemble(p, geos)
    print(f"[gpu-ensemble-blocks] {many.fluid_nodes()} nodes", flush=True)
    assert many.fluid_nodes() > 128 * 256
    out, fields = many.solve(check=100, tol=1e-5, max_steps=20000), many.fields()
    print(f"[gpu-ensemble-blocks] steps {sorted(set(out['steps'].tolist()))}", flush=True)
    for d in (0, 7, 23):
        one = ensemble.Ensemble(p, geos[d:d + 1])
        assert one.fluid_nodes() < 127 * 256
        alone = one.solve(check=100, tol=1e-5, max_steps=20000)
        assert alone["steps"][0] == out["steps"][d]
        assert alone["permeability"][0] == out["permeability"][d]
        assert np.array_equal(one.fields()[0], fields[d])
