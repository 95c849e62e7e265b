"""The block ILU(0) of polyhedra: rows with five to nine lower or upper
blocks (wide row entries, the eight-block kernels, and past eight the apply
from the block-CSR factor) whose couplings form triangles (the general factor),
against the numpy ILU(0)."""
import pytest

from polymeshes import hanging_nodes, one_merged
from test_gpu_ilu_apply import check_apply

pytestmark = pytest.mark.gpu

# more than 1024 cells: several partitions, several tiles of the natural order
MESHES = {f"{r + 1} blocks": (lambda r=r: hanging_nodes(8, 240 // r, r)) for r in (4, 5, 6, 7, 8)}


@pytest.mark.parametrize("order,precision,tol", [
    # the bounds of test_gpu_ilu_apply: ~1e3 eps of the precision
    ("natural", "fp64", 1e-12), ("natural", "mixed", 1e-4), ("partitioned", "fp64", 1e-12), ("partitioned", "mixed", 1e-4)])
@pytest.mark.parametrize("name", sorted(MESHES))
def test_one_direction_is_the_ilu_apply(name, order, precision, tol):
    # the diagonal grows with the row, as a matrix's does
    check_apply(MESHES[name](), 1, order, precision, tol, dominance=4.0 * int(name[0]))


# one polyhedron among quadrilaterals: the general factor packed into the tiles'
# and partitions' streams, its triangles inside one, across the sides of two and (the last) cut by a
# partition's side
@pytest.mark.parametrize("order,precision,tol", [
    ("natural", "fp64", 1e-12), ("natural", "mixed", 1e-4), ("partitioned", "fp64", 1e-12), ("partitioned", "mixed", 1e-4)])
@pytest.mark.parametrize("place", [(3, 3), (16, 15), (20, 19), (0, 27)])
def test_one_polyhedron(place, order, precision, tol):
    check_apply(one_merged(40, 40, *place), 2, order, precision, tol)
