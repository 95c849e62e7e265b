"""The GMRES orthogonalisations around the length up to which one workgroup
does a vector (4096 entries), against a sparse direct solve."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

from rhodst_amd import _capi, cases, meshgen
from rhodst_amd._abi import make_bcs, make_settings, make_thermo

pytestmark = pytest.mark.gpu


# 520, 4095 and 4100 unknowns, and two blocks of a long vector's grid stride
@pytest.mark.parametrize("nx,ny", [(13, 8), (9, 91), (10, 82), (300, 180)])
@pytest.mark.parametrize("gs", ["modified", "classical"])
def test_gmres_solves(nx, ny, gs):
    mesh = meshgen.box_2d(nx, ny, jitter=0.2)
    n, nI = mesh.n_cells, len(mesh.neighbour)
    rng = np.random.default_rng(nx)
    upper, lower = rng.uniform(-0.5, 0.5, (2, nI, 5, 5))
    own, nei = np.asarray(mesh.owner[:nI]), np.asarray(mesh.neighbour)
    diag = rng.uniform(-0.5, 0.5, (n, 5, 5)) + 8.0 * np.eye(5)
    b = rng.standard_normal((n, 5))
    kw = dict(n_directions=6, max_iter=8, min_iter=1, tolerance=1e-14, rel_tol=0.0, gram_schmidt=gs)
    patches = {p[0]: {"p": "zeroGradient", "T": "zeroGradient", "U": "zeroGradient"} for p in mesh.patches if p[1] != 3}
    spec = cases.CaseSpec("krylov", mesh, make_thermo(), make_bcs(mesh, patches), make_settings(**kw),
                          np.ones(n), np.ones(n), np.zeros((n, 3)))
    x, _ = _capi.DeviceCase(spec, _capi.DeviceMesh(mesh)).ldu_solve(diag, upper, lower, b, np.zeros((n, 5)))
    i = np.concatenate([np.arange(n), own, nei])
    j = np.concatenate([np.arange(n), nei, own])
    order = np.lexsort((j, i))
    A = sp.bsr_matrix((np.concatenate([diag, upper, lower])[order], j[order],
                       np.concatenate([[0], np.cumsum(np.bincount(i, minlength=n))])), shape=(5 * n, 5 * n))
    ref = spla.spsolve(A.tocsc(), b.ravel())
    # residual reduced to 1e-14 of the right-hand side's, condition number below 10
    assert np.abs(x.ravel() - ref).max() <= 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("nx,ny", [(13, 8), (40, 40)])  # one partition or tile, several
@pytest.mark.parametrize("kw", [dict(), dict(precision="mixed"),
                                dict(ilu_order="partitioned", precision="mixed", gram_schmidt="classical")],
                         ids=["fp64", "mixed", "partitioned mixed"])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_a_matrix_that_is_not_finite_shows_in_the_residuals(nx, ny, kw, bad):
    # 0 x inf and 0 x nan are nan: a solve from zero has no finite norm, whatever b is
    mesh = meshgen.box_2d(nx, ny)
    n, nI = mesh.n_cells, len(mesh.neighbour)
    rng = np.random.default_rng(nx)
    upper, lower = rng.uniform(-0.5, 0.5, (2, nI, 5, 5))
    diag = rng.uniform(-0.5, 0.5, (n, 5, 5)) + 8.0 * np.eye(5)
    patches = {p[0]: {"p": "zeroGradient", "T": "zeroGradient", "U": "zeroGradient"} for p in mesh.patches if p[1] != 3}
    spec = cases.CaseSpec("krylov", mesh, make_thermo(), make_bcs(mesh, patches),
                          make_settings(n_directions=4, min_iter=0, max_iter=2, **kw), np.ones(n), np.ones(n), np.zeros((n, 3)))
    dc = _capi.DeviceCase(spec, _capi.DeviceMesh(mesh))
    for b in (rng.standard_normal((n, 5)), np.zeros((n, 5))):
        u = upper.copy()
        u[nI // 2, 2, 3] = bad
        _, perf = dc.ldu_solve(diag, u, lower, b, np.zeros((n, 5)), mode=2)
        assert np.isnan(list(perf.initial_residual)).all() and np.isnan(list(perf.final_residual)).all()
        assert perf.n_iterations == 2 and not perf.converged
    # a finite one is converged at once for b = 0
    x, perf = dc.ldu_solve(diag, upper, lower, np.zeros((n, 5)), np.zeros((n, 5)), mode=2)
    assert not x.any() and perf.n_iterations == 0 and list(perf.initial_residual) == [0.0] * 5


# 820, 819, 182 and 169 cells: every remainder of 5 n by four, a tail of which the
# FP32 basis is padded with; 274 400 cells: the vectors past a grid stride of the
# four-wide loops (1.05 M entries), matrix and stream past 128 MiB in both
# precisions (non-temporal loads).  20 directions: three groups of eight of the
# multi-dot, five vectors at a time of the update.
@pytest.mark.parametrize("nx,ny", [(82, 10), (9, 91), (14, 13), (13, 13), (560, 490)])
@pytest.mark.parametrize("kw", [dict(gram_schmidt="modified"), dict(gram_schmidt="classical"),
                                dict(gram_schmidt="modified", precision="mixed"),
                                dict(gram_schmidt="classical", precision="mixed")],
                         ids=lambda kw: "-".join(kw.values()))
def test_residual_of_a_converged_solve(nx, ny, kw):
    mesh = meshgen.box_2d(nx, ny)
    n, nI = mesh.n_cells, len(mesh.neighbour)
    rng = np.random.default_rng(ny)
    upper, lower = rng.uniform(-0.5, 0.5, (2, nI, 5, 5))
    own, nei = np.asarray(mesh.owner[:nI]), np.asarray(mesh.neighbour)
    # coupled strongly enough that a cycle needs its 20 directions
    diag = rng.uniform(-0.5, 0.5, (n, 5, 5)) + 4.0 * np.eye(5)
    b = rng.standard_normal((n, 5))
    patches = {p[0]: {"p": "zeroGradient", "T": "zeroGradient", "U": "zeroGradient"} for p in mesh.patches if p[1] != 3}
    st = make_settings(n_directions=20, max_iter=8, min_iter=1, tolerance=1e-15, rel_tol=0.0, ilu_order="partitioned", **kw)
    spec = cases.CaseSpec("krylov", mesh, make_thermo(), make_bcs(mesh, patches), st, np.ones(n), np.ones(n), np.zeros((n, 3)))
    x, perf = _capi.DeviceCase(spec, _capi.DeviceMesh(mesh)).ldu_solve(diag, upper, lower, b, np.zeros((n, 5)))
    r = b - np.einsum("nij,nj->ni", diag, x)
    np.subtract.at(r, own, np.einsum("nij,nj->ni", upper, x[nei]))
    np.subtract.at(r, nei, np.einsum("nij,nj->ni", lower, x[own]))
    # rounding of the residual itself: 25 products of about |b| per entry
    assert np.linalg.norm(r) <= 1e-13 * np.linalg.norm(b)
    # an FP32 basis loses what FP64 has, not cycles: 1e-5 and more per cycle of 20 directions
    assert perf.n_iterations <= 5


@pytest.mark.parametrize("order,precision", [("natural", "fp64"), ("natural", "mixed"), ("partitioned", "fp64"),
                                             ("partitioned", "mixed")])
@pytest.mark.parametrize("nx,ny", [(13, 8), (40, 40)])  # one partition or tile, several that wait for each other
def test_a_singular_pivot_block_is_an_error(nx, ny, order, precision):
    mesh = meshgen.box_2d(nx, ny)
    n, nI = mesh.n_cells, len(mesh.neighbour)
    rng = np.random.default_rng(nx)
    upper, lower = rng.uniform(-0.5, 0.5, (2, nI, 5, 5))
    diag = rng.uniform(-0.5, 0.5, (n, 5, 5)) + 8.0 * np.eye(5)
    b = rng.standard_normal((n, 5))
    patches = {p[0]: {"p": "zeroGradient", "T": "zeroGradient", "U": "zeroGradient"} for p in mesh.patches if p[1] != 3}
    spec = cases.CaseSpec("krylov", mesh, make_thermo(), make_bcs(mesh, patches),
                          make_settings(n_directions=4, ilu_order=order, precision=precision),
                          np.ones(n), np.ones(n), np.zeros((n, 3)))
    dc = _capi.DeviceCase(spec, _capi.DeviceMesh(mesh))
    x, _ = dc.ldu_solve(diag, upper, lower, b, np.zeros((n, 5)))
    # cell 0 has no lower neighbour: its pivot block is the diagonal block
    zero = diag.copy()
    zero[0] = 0.0
    with pytest.raises(_capi.RdstError, match="singular pivot"):
        dc.ldu_solve(zero, upper, lower, b, np.zeros((n, 5)))
    # and the system before it has the same solution after it
    assert np.array_equal(dc.ldu_solve(diag, upper, lower, b, np.zeros((n, 5)))[0], x)
