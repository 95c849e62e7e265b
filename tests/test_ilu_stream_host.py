"""The ILU(0) record streams and the tiles of the natural-order sweeps,
replayed on the CPU (tests/host/ilu_stream_check.cpp) over meshes of every
numbering: structured, curvilinear with a wake cut, hybrid, tetrahedra, and
the same cells numbered at random."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from polymeshes import hanging_nodes, one_merged, triangles
from rhodst_amd import DeviceMesh, _capi, meshgen
from rhodst_amd._abi import MeshDesc, rdst_mesh_desc

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def replay_lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host") / "ilu_stream_check.so")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I", f"{rocm}/include",
                    "-I", os.path.join(HERE, "..", "include"), os.path.join(HERE, "host", "ilu_stream_check.cpp"),
                    "-L", f"{rocm}/lib", "-lamdhip64", "-pthread", f"-Wl,-rpath,{rocm}/lib", "-o", so], check=True)
    lib = C.CDLL(so)
    for f in (lib.ilu_stream_check, lib.ilu_plan_retry):
        f.argtypes = [C.POINTER(rdst_mesh_desc), C.c_int, C.c_int, C.c_char_p, C.c_int]
    return lib


def shuffled(mesh, seed):
    """The same cells in a random order (owner/neighbour of a face swapped to
    keep the lower cell its owner, faces in upper-triangular order)."""
    rng = np.random.default_rng(seed)
    p = rng.permutation(mesh.n_cells)
    own, nei = p[np.asarray(mesh.owner)], p[np.asarray(mesh.neighbour)]
    nI = len(nei)
    fp = [list(mesh.face_points[mesh.face_offsets[f]:mesh.face_offsets[f + 1]]) for f in range(len(own))]
    for f in range(nI):
        if own[f] > nei[f]:
            own[f], nei[f] = nei[f], own[f]
            fp[f] = fp[f][:1] + fp[f][:0:-1]
    order = np.concatenate([np.lexsort((nei, own[:nI])), np.arange(nI, len(own))])
    fp = [fp[f] for f in order]
    import copy
    m = copy.copy(mesh)
    m.owner, m.neighbour = own[order].astype(np.int32), nei[order[:nI]].astype(np.int32)
    m.face_points = np.concatenate([np.asarray(q) for q in fp]).astype(np.int32)
    m.face_offsets = np.concatenate([[0], np.cumsum([len(q) for q in fp])]).astype(np.int32)
    return m


MESHES = {
    "one cell": lambda: meshgen.box_2d(1, 1),
    "line": lambda: meshgen.channel_1d(2500),
    "box 33x31": lambda: meshgen.box_2d(33, 31, jitter=0.2),  # 1023 cells: one tile
    "box 25x41": lambda: meshgen.box_2d(25, 41, jitter=0.2),  # 1025: several
    "box 150x70": lambda: meshgen.box_2d(150, 70, jitter=0.2),
    "step": lambda: meshgen.forward_step(120, 40),
    "hybrid airfoil": lambda: meshgen.hybrid_airfoil(n_surf=80, n_layers=16, first_cell=2e-5, far=8.0),
    "wing": lambda: meshgen.swept_wing(n_wake=13, n_surf=30, n_normal=21, n_span_wing=9, n_span_out=5, n_layers=8),
    "wing tiles": lambda: meshgen.swept_wing(n_wake=6, n_surf=16, n_normal=16, n_span_wing=8, n_span_out=4, n_layers=8,
                                             order="tiles"),
    "tets": lambda: meshgen.tet_prism_box(11, 13, 12, prism_layers=3, jitter=0.1),
    "box shuffled": lambda: shuffled(meshgen.box_2d(60, 45, jitter=0.2), 1),
    "tets shuffled": lambda: shuffled(meshgen.tet_prism_box(7, 6, 8, prism_layers=3, jitter=0.1), 2),
    # rows of up to eight blocks, couplings in triangles
    "polyhedra": lambda: hanging_nodes(9, 40, 7),
    "polyhedra shuffled": lambda: hanging_nodes(9, 100, 3, seed=1),
    "one polyhedron": lambda: one_merged(40, 40, 16, 15),
}


@pytest.mark.parametrize("name", sorted(MESHES))
def test_streams_and_tiles(replay_lib, name):
    md = MeshDesc(MESHES[name]())
    what = C.create_string_buffer(256)
    for fp32 in (0, 1):
        for natural in (0, 1):
            rc = replay_lib.ilu_stream_check(C.byref(md.desc), fp32, natural, what, 256)
            assert rc == 0, (name, fp32, natural, what.value.decode())


@pytest.mark.parametrize("cells", [1, 33_554_431, 33_554_432, 67_108_864, 120_000_000])
@pytest.mark.parametrize("ent", [16, 32])
def test_row_entries_of_large_meshes(replay_lib, cells, ent):
    # the last of two entries per cell, at the sizes where its byte offset passes 31 and 32 bits
    replay_lib.ilu_entry_unit.restype = C.c_longlong
    row = 2 * cells - 1
    assert 16 * replay_lib.ilu_entry_unit(row, ent) == row * ent


@pytest.mark.parametrize("cells", [1, 85_899_345, 85_899_346, 140_000_000])
@pytest.mark.parametrize("nv", [5, 25])
def test_halo_values_of_large_meshes(replay_lib, cells, nv):
    # the last value of the last cell, at the sizes where 25 per cell pass 31 bits
    replay_lib.ilu_cell_value.restype = C.c_longlong
    assert replay_lib.ilu_cell_value(cells - 1, nv, nv - 1) == nv * cells - 1


@pytest.mark.parametrize("name", ["box 25x41", "tets shuffled"])
@pytest.mark.parametrize("natural", [0, 1])
@pytest.mark.parametrize("fp32", [0, 1])
def test_plan_after_running_out_of_memory(replay_lib, name, natural, fp32):
    md = MeshDesc(MESHES[name]())
    what = C.create_string_buffer(256)
    rc = replay_lib.ilu_plan_retry(C.byref(md.desc), fp32, natural, what, 256)
    assert rc == 0, what.value.decode()


def test_one_upload_for_all_threads(replay_lib):
    md = MeshDesc(MESHES["box 25x41"]())
    replay_lib.mesh_upload_mallocs.argtypes = [C.POINTER(rdst_mesh_desc), C.c_int]
    one = replay_lib.mesh_upload_mallocs(C.byref(md.desc), 1)
    assert one > 10 and replay_lib.mesh_upload_mallocs(C.byref(md.desc), 8) == one


def plan_numbers(lib, mesh, natural, fp32=0):
    out = (C.c_int * 4)()
    lib.ilu_plan_numbers.argtypes = [C.POINTER(rdst_mesh_desc), C.c_int, C.c_int, C.POINTER(C.c_int)]
    lib.ilu_plan_numbers.restype = None
    md = MeshDesc(mesh)
    lib.ilu_plan_numbers(C.byref(md.desc), fp32, natural, out)
    return list(out)


@pytest.mark.parametrize("name,tiles", [
    # one tile, and numberings with many levels and thin halos
    ("one cell", True), ("box 33x31", True), ("line", True), ("box 150x70", True), ("hybrid airfoil", True), ("wing", True),
    ("wing tiles", True),
    # a dozen levels
    ("box shuffled", False), ("tets shuffled", False)])
def test_tiles_where_they_pay(replay_lib, name, tiles):
    kmax, _, n, ok = plan_numbers(replay_lib, MESHES[name](), natural=1)
    assert bool(ok) == tiles and (kmax > 0) == tiles
    assert (n == 1) == (name in ("one cell", "box 33x31"))


@pytest.mark.parametrize("parts,levels,columns,rows,memory", [
    # the sweeps timed both ways: partitions, mean levels, columns per row, rows of the largest
    (2048, 53, 6, 990, False), (4096, 53, 6, 958, False), (256, 89, 6, 704, False), (4096, 89, 6, 975, True),
    (256, 89, 8, 704, False), (1024, 100, 8, 875, False), (2048, 104, 8, 879, True),
    # two partitions per CU
    (16384, 40, 6, 563, False), (4096, 63, 4, 977, False)])
def test_gauss_seidel_form(replay_lib, parts, levels, columns, rows, memory):
    replay_lib.sa_sgs_from_memory.argtypes = [C.c_int, C.c_double, C.c_int, C.c_int]
    lds = (8 * (columns + 3) + 2 * (columns + 1)) * rows
    assert bool(replay_lib.sa_sgs_from_memory(parts, levels, columns, lds)) == memory


# the polyhedron inside a tile and a partition, and at the sides of several (tiles of
# 16 x 8 cells, the second row and column of partitions from 20 on); the last two
# triangles are cut by a partition's side, which leaves its factor a chain
PLACES = [(3, 3), (15, 3), (16, 3), (4, 7), (15, 7), (16, 15), (19, 19), (20, 19), (19, 20), (20, 5), (38, 37),
          (0, 27), (39, 10)]


@pytest.mark.parametrize("mesh", [lambda: hanging_nodes(9, 40, 7), lambda: hanging_nodes(9, 100, 3, seed=1)] +
                         [lambda p=p: one_merged(40, 40, *p) for p in PLACES],
                         ids=["polyhedra", "polyhedra shuffled"] + [f"{i},{j}" for i, j in PLACES])
def test_chain_factor_only_without_triangles(replay_lib, mesh):
    pm = mesh()
    part = DeviceMesh(pm).get_int(_capi.M_PARTITION)
    lower = np.zeros(pm.n_cells, dtype=int)
    inside = part[pm.owner[:len(pm.neighbour)]] == part[pm.neighbour]
    np.add.at(lower, pm.neighbour[inside], 1)
    _, chain, n, _ = plan_numbers(replay_lib, pm, natural=0)
    assert n == part.max() + 1 >= 2
    assert (chain > 0) == (not triangles(pm, part) and lower.max() <= 4)
    assert triangles(pm)
    kmax, chain, n, ok = plan_numbers(replay_lib, pm, natural=1)
    assert chain == 0 and n > 1 and bool(kmax) == bool(ok)
