"""Fields of structures to and from the device's component arrays
(rdst_case_get / rdst_case_put), at sizes about one 256-thread block and past
one staging piece."""
import numpy as np
import pytest

from rhodst_amd import DeviceCase, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(1, 1), (17, 15), (1300, 1291)])
def test_momentum_round_trip(nx, ny):
    spec = cases.box_farfield_case(nx=nx, ny=ny, jitter=0.0)
    dc = DeviceCase(spec)
    rho, U = dc.get(0), dc.get(5)
    assert np.array_equal(U, spec.U0)
    assert np.array_equal(dc.get(1), rho[:, None] * U)  # 40 MB at the largest size
    v = np.random.default_rng(1).standard_normal((nx * ny, 3))
    dc.put(1, v)
    assert np.array_equal(dc.get(1), v)
    # five components, 67 MB at the largest size: more than one staging piece
    dc.flux_residual()
    R = dc.get(8)
    assert R.shape == (nx * ny, 5) and np.isfinite(R).all()
    assert np.isclose(np.sqrt((R ** 2).sum()), dc.set_courant(), rtol=1e-12)
