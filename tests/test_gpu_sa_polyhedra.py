"""The Spalart-Allmaras Gauss-Seidel sweep on polyhedra: rows with six, eight and
ten columns in a partition (the six- and eight-column forms in LDS, and the one
from memory), against the oracle given the same partition."""
import numpy as np
import pytest

from rhodst_amd import DeviceCase, _capi, cases, meshgen
from polymeshes import hanging_nodes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ratio", [2, 3, 4])
def test_partitioned_sweep_parity(oracle, monkeypatch, ratio):
    print(f"[SA polyhedra] {ratio}", flush=True)
    mesh = hanging_nodes(12, 240 // ratio, ratio)
    monkeypatch.setattr(meshgen, "box_2d", lambda *a, **k: mesh)
    spec = cases.box_sa_case("SAneg", turb_kw={"rel_tol": 1e-3, "tolerance": 1e-12, "min_iter": 3})
    dc = DeviceCase(spec)
    part = dc.mesh.get_int(_capi.M_SA_PARTITION)
    assert part.max() >= 1
    oc = oracle.OracleCase(spec)
    oc.set_sa_partition(part)
    oc.flux_residual()
    dc.flux_residual()
    po = oc.turbulence_correct()
    pd = dc.turbulence_correct()
    assert po.n_iterations >= 3 and pd.n_iterations == po.n_iterations
    for f in (29, 30):  # nuTilda and mut, the bound of the same test on quadrilaterals
        d, o = dc.get(f), oc.get(f)
        assert np.abs(d - o).max() <= 1e-10 * np.abs(o).max()
