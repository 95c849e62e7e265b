"""Meshes of polyhedra for the tests of the ILU(0): cells of the generators'
meshes merged and relabelled."""
import copy

import numpy as np

from rhodst_amd import meshgen


def relabelled(mesh, label):
    """Cell c becomes part of cell label[c] (labels 0 .. max): faces inside a
    cell are dropped, the others get the lower label as their owner, in
    upper-triangular order."""
    label = np.asarray(label)
    nI = len(mesh.neighbour)
    own, nei = label[np.asarray(mesh.owner)], label[np.asarray(mesh.neighbour)]
    flip = own[:nI] > nei
    lo, hi = np.minimum(own[:nI], nei), np.maximum(own[:nI], nei)
    inner = np.nonzero(lo != hi)[0]
    faces = np.concatenate([inner[np.lexsort((hi[inner], lo[inner]))], np.arange(nI, len(own))])
    fp = []
    for f in faces:
        p = list(mesh.face_points[mesh.face_offsets[f]:mesh.face_offsets[f + 1]])
        fp.append(p[:1] + p[:0:-1] if f < nI and flip[f] else p)
    m = copy.copy(mesh)
    m.owner = np.where(faces < nI, np.append(lo, np.zeros(len(own) - nI, dtype=lo.dtype))[faces], own[faces]).astype(np.int32)
    m.neighbour = hi[faces[:len(inner)]].astype(np.int32)
    m.face_points = np.concatenate([np.asarray(p) for p in fp]).astype(np.int32)
    m.face_offsets = np.concatenate([[0], np.cumsum([len(p) for p in fp])]).astype(np.int32)
    m.n_cells = int(label.max()) + 1
    m.patches = [(name, kind, start - (nI - len(inner)), size) for name, kind, start, size in mesh.patches]
    return m


def hanging_nodes(nx, ny, ratio, seed=None):
    """A 2-D box whose odd columns have ny cells and whose even ones ny x ratio:
    a coarse cell has ratio neighbours on either side, each coupled with the
    next, so the couplings form triangles; numbered by column (coarse rows have
    ratio + 1 lower and upper neighbours) or, with a seed, at random."""
    mesh = meshgen.box_2d(nx, ny * ratio)
    i, j = np.arange(mesh.n_cells) % nx, np.arange(mesh.n_cells) // nx
    key = i * (ny * ratio) + np.where(i % 2 == 1, j // ratio * ratio, j)
    label = np.unique(key, return_inverse=True)[1]
    if seed is not None:
        label = np.random.default_rng(seed).permutation(label.max() + 1)[label]
    return relabelled(mesh, label)


def one_merged(nx, ny, i, j):
    """A 2-D box with cells (i, j) and (i, j + 1) merged into one: its couplings
    form two triangles (one at a side), with the two cells left and right of it."""
    mesh = meshgen.box_2d(nx, ny)
    label = np.arange(mesh.n_cells)
    label[i + nx * (j + 1)] = i + nx * j
    return relabelled(mesh, np.unique(label, return_inverse=True)[1])


def triangles(mesh, part=None):
    """Whether three cells (of one part) are coupled pairwise."""
    nb = [set() for _ in range(mesh.n_cells)]
    for a, b in zip(mesh.owner, mesh.neighbour):
        if part is None or part[a] == part[b]:
            nb[a].add(b)
            nb[b].add(a)
    return any(nb[a] & nb[b] for a in range(mesh.n_cells) for b in nb[a] if b > a)
