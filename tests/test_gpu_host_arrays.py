"""Fields of structures to and from the device's component arrays
(rdst_case_get / rdst_case_put), at sizes about one 256-thread block and past
one staging piece."""
import numpy as np
import pytest
import torch

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


def test_the_first_read_back_allocates_nothing():
    # 480 k cells: the staging of R (19 MB) shows in the device's free memory
    spec = cases.box_farfield_case(nx=800, ny=600, jitter=0.0)
    dc = DeviceCase(spec)
    dc.flux_residual()
    free = torch.cuda.mem_get_info()[0]
    R = dc.get(8)
    dc.put(1, dc.get(1))
    assert torch.cuda.mem_get_info()[0] == free
    assert np.array_equal(R, dc.get(8))
