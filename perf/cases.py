"""Performance cases of the implicit step: what a user of the library runs,
through the C-ABI and its ctypes binding, over the range of sizes and options.

A case is a dict of plain values.  ``call`` says which entry points one pass
goes through:

  iterate  rdst_iterate (Single::iterate) on a resident case, then W (and
           nuTilda) read back: the time loop of a run
  flux     rdst_flux_residual on a resident state, then R and phi read back:
           the residual evaluation of an adapter that keeps its own solver
  ldu      rdst_ldu_solve on a system the caller assembled in host memory
  adjoint  rdst_adjoint_linearise at a viscous state and one product J^T x

``path`` is the linear solver a user picks: "plain" (FP64, natural-order
ILU(0), modified Gram-Schmidt: the reference's own algorithm and the default
settings), "fp64" (FP64, partitioned ILU(0), classical Gram-Schmidt), "mixed"
(the same in FP32 inside an FP64 defect correction).
"""
import functools
import math

import numpy as np
import torch

from rhodst_amd import DeviceCase, DeviceMesh, cases, lib, meshgen
from rhodst_amd._abi import dptr

PATHS = {
    "plain": {},
    "fp64": dict(ilu_order="partitioned", gram_schmidt="classical"),
    "mixed": dict(ilu_order="partitioned", gram_schmidt="classical", precision="mixed"),
}
F_R, F_W, F_PHI, F_NUT = 8, 9, 12, 29


def listed():
    return [
        # the smallest runs: a few hundred cells with the default settings (a
        # smoke test, a parameter study in 2-D), bound by latency and launches
        dict(name="forward_step_small_plain", call="iterate", mesh="forward_step", nx=30, ny=10, scheme="AUSM+",
             path="plain"),
        # the Mach-3 forward step at its tutorial size through the fast path
        dict(name="forward_step_mixed", call="iterate", mesh="forward_step", nx=120, ny=40, scheme="AUSM+",
             path="mixed"),
        # the RAE2822 tutorial with the fvSchemes and fvSolution it ships:
        # limited reconstruction, BiCGStab + natural-order ILU(0), stock SA
        dict(name="rae2822_plain", call="iterate", mesh="rae2822", scheme="Kurganov", path="plain"),
        # 2-D RANS on the hybrid quad/triangle airfoil mesh, about 2e5 cells
        dict(name="airfoil_mixed", call="iterate", mesh="airfoil", n_surf=400, scheme="HLLC", turbulence="SAneg",
             path="mixed"),
        # the headline workload: the 2.03 M-cell swept wing, SA with
        # rotation-curvature correction, mixed precision
        dict(name="wing_2m_mixed", call="iterate", mesh="wing", n_wake=48, n_surf=128, n_normal=96, n_span_wing=44,
             n_span_out=16, scheme="AUSM+up", turbulence="SARC2", path="mixed"),
        # a mid-size wing with ragged dimensions in FP64
        dict(name="wing_400k_fp64", call="iterate", mesh="wing", n_wake=29, n_surf=71, n_normal=53, n_span_wing=27,
             n_span_out=11, scheme="AUSM+up", turbulence="SARC2", path="fp64"),
        # the reference's own algorithm on a wing
        dict(name="wing_320k_plain", call="iterate", mesh="wing", n_wake=24, n_surf=64, n_normal=48, n_span_wing=22,
             n_span_out=16, scheme="AUSM+up", turbulence="SARC2", path="plain"),
        # tetrahedra over prism layers with Kurganov and SAneg, 1.15 M cells
        dict(name="tet_prism_mixed", call="iterate", mesh="tet_prism", nx=60, ny=60, nz=60, layers=10,
             scheme="Kurganov", turbulence="SAneg", path="mixed"),
        # Newton-Krylov: the exact-Jacobian operator on an inviscid wing
        dict(name="wing_newton_mixed", call="iterate", mesh="wing", n_wake=24, n_surf=64, n_normal=48, n_span_wing=22,
             n_span_out=16, scheme="AUSM+up", turbulence="", path="mixed", jacobian="exact"),
        # residual evaluations of a viscous wing with R and phi on the host
        dict(name="wing_flux", call="flux", mesh="wing", n_wake=31, n_surf=86, n_normal=64, n_span_wing=29,
             n_span_out=11, scheme="AUSM+up", turbulence="SARC2", path="fp64"),
        # a caller's own LDU system (foam's matrix) solved on the GPU
        dict(name="wing_ldu_fp64", call="ldu", mesh="wing", n_wake=13, n_surf=48, n_normal=37, n_span_wing=19,
             n_span_out=7, scheme="AUSM+up", turbulence="", path="fp64"),
        # sensitivities: the exact viscous linearisation and a transposed product
        dict(name="airfoil_adjoint", call="adjoint", mesh="airfoil", n_surf=200, scheme="HLLC", turbulence="SAneg",
             path="fp64"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["forward_step", "airfoil", "wing", "wing", "tet_prism", "newton", "flux", "ldu", "adjoint"])
    if kind == "forward_step":
        k = _log_int(rng, 2, 12)  # nx = 3 ny, ny a multiple of 5 (meshgen.forward_step)
        return dict(call="iterate", mesh="forward_step", nx=15 * k, ny=5 * k,
                    scheme=rng.choice(["AUSM+", "AUSM+up", "HLL", "HLLC", "HLLCP", "Kurganov"]),
                    path=rng.choice(["plain", "mixed", "fp64"]))
    if kind in ("airfoil", "adjoint"):
        n = _log_int(rng, 80, 400 if kind == "airfoil" else 220)
        return dict(call="iterate" if kind == "airfoil" else "adjoint", mesh="airfoil", n_surf=n + n % 2,
                    scheme=rng.choice(["HLLC", "AUSM+up", "Kurganov"]), turbulence=rng.choice(["SAneg", "SARC2"]),
                    path=rng.choice(["mixed", "fp64"]) if kind == "airfoil" else "fp64")
    if kind == "tet_prism":
        n = [_log_int(rng, lo, 60) for lo in (8, 8, 24)]
        return dict(call="iterate", mesh="tet_prism", nx=n[0], ny=n[1], nz=n[2], layers=max(6, n[2] // rng.randint(4, 5)),
                    scheme=rng.choice(["Kurganov", "HLLC"]), turbulence=rng.choice(["SAneg", "SARC2"]),
                    path=rng.choice(["mixed", "fp64"]))
    # wings from about 1e4 cells to the headline size
    big = {"wing": 1.0, "newton": 0.55, "flux": 1.0, "ldu": 0.45}[kind]
    path = rng.choice(["mixed", "mixed", "fp64", "plain"]) if kind == "wing" else rng.choice(["mixed", "fp64"])
    if path == "plain":
        big = 0.5
    f = math.exp(rng.uniform(math.log(0.2), math.log(big)))
    j = lambda v, least: max(least, int(round(v * f * rng.uniform(0.9, 1.0))))  # noqa: E731
    turb = rng.choice(["SARC2", "SAneg"]) if kind in ("wing", "flux") else ""
    c = dict(call="iterate" if kind in ("wing", "newton") else kind, mesh="wing", n_wake=j(48, 6), n_surf=j(128, 16),
             n_normal=j(96, 40), n_span_wing=j(44, 8), n_span_out=j(16, 4), scheme=rng.choice(["AUSM+up", "HLLC"]),
             turbulence=turb, path="fp64" if kind == "flux" else path)
    if kind == "newton":
        c["jacobian"] = "exact"
    return c


# ---------------------------------------------------------------- meshes
_SIZES = ("nx", "ny", "nz", "layers", "n_surf", "n_wake", "n_normal", "n_span_wing", "n_span_out")


@functools.lru_cache(maxsize=3)
def _polymesh(kind, sizes):
    s = dict(sizes)
    if kind == "forward_step":
        return meshgen.forward_step(s["nx"], s["ny"])
    if kind == "rae2822":
        return meshgen.polymesh_from_npz(cases.RAE2822_MESH)
    if kind == "airfoil":
        # a coarser surface goes with a thicker first cell and fewer wall layers
        thick = (400 / s["n_surf"]) ** 1.4
        return meshgen.hybrid_airfoil(n_surf=s["n_surf"], first_cell=2e-6 * thick,
                                      n_layers=40 - round(math.log(thick) / math.log(1.15)))
    if kind == "tet_prism":
        return meshgen.tet_prism_box(s["nx"], s["ny"], s["nz"], prism_layers=s["layers"], lx=1.0, ly=0.6, lz=0.4,
                                     first=2e-5, jitter=0.1)
    return meshgen.swept_wing(**s)


@functools.lru_cache(maxsize=3)
def _mesh(kind, sizes):
    """The mesh handle (and the wall distance of a viscous case), made once
    per mesh as a program that runs several cases on one mesh does."""
    pm = _polymesh(kind, sizes)
    dm = DeviceMesh(pm)
    return pm, dm, (dm.wall_distance() if kind != "forward_step" else None)


def _sizes(case):
    return tuple((k, case[k]) for k in _SIZES if k in case)


# ---------------------------------------------------------------- states
def _settings(case, path):
    kw = dict(PATHS[path])
    if case["mesh"] == "forward_step":
        kw.update(initial_co=3.0, min_co=3.0, max_co=3.0)
    elif case["mesh"] == "rae2822":
        kw.update(max_co=20.0)  # a point on the tutorial's ramp 1 -> 500
    elif case["mesh"] == "tet_prism":
        kw.update(n_directions=30, rel_tol=1e-2, max_iter=1)
    return kw


def _make(case, **kw):
    """The case of the framework's own generators on the shared mesh."""
    pm, dm, wd = _mesh(case["mesh"], _sizes(case))
    turb = case.get("turbulence") or None
    if case["mesh"] == "forward_step":
        spec = cases.forward_step_case(case["nx"], case["ny"], case["scheme"], **kw)
    elif case["mesh"] == "rae2822":
        spec = cases.rae2822_case(case["scheme"], mesh=pm, wall_dist=wd, **kw)
    elif case["mesh"] == "airfoil":
        spec = cases.airfoil_case(case["scheme"], turbulence=turb, mesh=pm, wall_dist=wd, **kw)
    elif case["mesh"] == "tet_prism":
        spec = cases.tet_prism_case(turb, case["scheme"], mesh=pm, perturb=0.0, wall_dist=wd, **kw)
    else:
        spec = cases.swept_wing_case(case["scheme"], mesh=pm, wall_dist=wd, turbulence=turb, **kw)
    return spec, dm


@functools.lru_cache(maxsize=3)
def _developed(items):
    """p, T, U (and nuTilda) after the first steps of an FP64 run from the
    uniform start: the field a restarted run reads from its time directory."""
    case = dict(items)
    spec, dm = _make(case, **_settings(case, "fp64"))
    dc = DeviceCase(spec, dm)
    dc.iterate({"forward_step": 800, "airfoil": 15}.get(case["mesh"], 30))
    return dc.get(3), dc.get(4), dc.get(5), (dc.get(F_NUT) if spec.turbulence is not None else None)


def _spec(case, seed):
    """The case restarted from its developed field with a small seeded
    disturbance of every cell."""
    kw = _settings(case, case["path"])
    if case["mesh"] == "rae2822":
        kw.update(initial_co=20.0, min_co=20.0)  # the field is past the start of the ramp
    if case.get("jacobian"):
        kw.update(jacobian=case["jacobian"], initial_co=2.0, max_co=100.0, update_limit=0.2)
    p, T, U, nut = _developed(tuple((k, v) for k, v in sorted(case.items()) if k not in ("name", "call", "path", "jacobian")))
    spec, dm = _make(case, **kw)
    rng = np.random.default_rng(seed)
    n = len(p)
    spec.p0 = p * (1 + 1e-5 * rng.uniform(-1, 1, n))
    spec.T0 = T * (1 + 1e-5 * rng.uniform(-1, 1, n))
    spec.U0 = U * (1 + 1e-5 * rng.uniform(-1, 1, (n, 1)))
    if nut is not None:
        t, bcs, wd, _ = spec.turbulence
        spec.turbulence = (t, bcs, wd, nut * (1 + 1e-5 * rng.uniform(-1, 1, n)))
    return spec, dm


def _host(*shape):
    """A pinned host array, as a program that reads fields back every step keeps."""
    t = torch.empty(shape, dtype=torch.float64)
    return t.pin_memory() if torch.cuda.is_available() else t


def _get(dc, field, out):
    rc = lib().rdst_case_get(dc.h, field, dptr(out.numpy()))
    if rc:
        raise RuntimeError(lib().rdst_last_error().decode())
    return out


def _ldu_system(case, seed):
    """A block system of the kind an implicit step gives, in foam's LDU
    order: random coupling blocks of unequal size per face, a diagonal that
    dominates them by a pseudo-time term, and a right-hand side."""
    pm = _polymesh(case["mesh"], _sizes(case))
    nI, n = len(pm.neighbour), pm.n_cells
    g = torch.Generator().manual_seed(int(seed))
    scale = 0.1 + torch.rand(nI, 1, 1, generator=g, dtype=torch.float64)
    upper = scale * (torch.rand(nI, 5, 5, generator=g, dtype=torch.float64) - 0.5)
    lower = scale * (torch.rand(nI, 5, 5, generator=g, dtype=torch.float64) - 0.5)
    own = torch.as_tensor(np.asarray(pm.owner[:nI], dtype=np.int64))
    nei = torch.as_tensor(np.asarray(pm.neighbour, dtype=np.int64))
    eye = torch.eye(5, dtype=torch.float64)
    diag = 0.4 * eye + 0.2 * (torch.rand(n, 5, 5, generator=g, dtype=torch.float64) - 0.5)
    for s in (own, nei):
        diag.index_add_(0, s, scale * eye)
    b = torch.rand(n, 5, generator=g, dtype=torch.float64) - 0.5
    return diag, upper, lower, own, nei, b


def prepare(case, seed):
    s = {"call": case["call"]}
    if case["call"] == "ldu":
        spec, dm = _make(case, **_settings(case, case["path"]))
        # a few restart cycles to the accuracy an implicit step asks for
        spec.settings.rel_tol, spec.settings.max_iter = 1e-6, 10
        diag, upper, lower, _, _, b = _ldu_system(case, seed)
        s.update(dc=DeviceCase(spec, dm), diag=diag.numpy(), upper=upper.numpy(), lower=lower.numpy(), b=b.numpy(),
                 x=np.zeros(b.shape))
        return s
    spec, dm = _spec(case, seed)
    dc = s["dc"] = DeviceCase(spec, dm)
    n, nf = dc.n, dc.nI + dc.nB
    dc.iterate(1)  # a program that has run before keeps the solver's workspace; back to the state
    dc.set_state(spec.p0, spec.T0, spec.U0)
    if spec.turbulence is not None:
        dc.set_turbulence(*spec.turbulence)
    if case["call"] == "iterate":
        s["W"] = _host(n, 5)
        if spec.turbulence is not None:
            s["nut"] = _host(n)
    elif case["call"] == "flux":
        s["R"], s["phi"] = _host(n, 5), _host(nf)
    else:
        s["x"] = np.random.default_rng(seed).standard_normal((n, 5))
    return s


def run(s):
    dc = s["dc"]
    if s["call"] == "iterate":
        out = {"res": dc.iterate(1), "W": _get(dc, F_W, s["W"])}
        if "nut" in s:
            out["nut"] = _get(dc, F_NUT, s["nut"])
        return out
    if s["call"] == "flux":
        dc.flux_residual()
        return {"R": _get(dc, F_R, s["R"]), "phi": _get(dc, F_PHI, s["phi"])}
    if s["call"] == "ldu":
        return {"x": dc.ldu_solve(s["diag"], s["upper"], s["lower"], s["b"], s["x"])[0]}
    dc.adjoint_linearise()
    return {"y": dc.adjoint_apply(s["x"], transpose=True)}


# ---------------------------------------------------------------- work
def work(case):
    """What one pass cannot do without.  N cells, F internal faces: the state
    in and out and the face geometry once; the matrix read per product and its
    factor per application; the Krylov basis once per orthogonalisation."""
    pm = _polymesh(case["mesh"], _sizes(case))
    N, F = pm.n_cells, len(pm.neighbour)
    nnzb, s = N + 2 * F, 4 if case["path"] == "mixed" else 8
    face, state = 80.0 * F, 80.0 * N
    if case["call"] == "flux":
        return {"bytes": face + state + 120.0 * N + 8.0 * F, "flops": 700.0 * F}
    if case["call"] == "adjoint":
        return {"bytes": face + state + 2 * 200.0 * (N + 6.0 * F), "flops": 5 * 2 * 700.0 * F * 4}
    its = {"forward_step": 20, "rae2822": 200}.get(case["mesh"], 30)
    basis = 5.0 * N * s * (its / 2 if case["mesh"] != "rae2822" else 6)
    mat = 25.0 * s * nnzb
    b = face + state + mat + its * (2 * mat + basis)
    if case["call"] == "ldu":
        b += 200.0 * nnzb
    return {"bytes": b, "flops": its * (100.0 * nnzb + 4 * basis / s) + 1500.0 * F}


# ---------------------------------------------------------------- exact
def exact(case, seed):
    """The solution of the caller's system in 64 bits (restarted BiCGStab with
    the inverted diagonal blocks to rounding error); the other calls return
    64-bit fields after a nonlinear step, which have no short closed form."""
    if case["call"] != "ldu":
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    diag, upper, lower, own, nei, b = (t.to(dev) for t in _ldu_system(case, seed))
    dinv = torch.linalg.inv(diag)

    def mul(m, v):
        return (m * v[:, None, :]).sum(-1)

    def A(v):
        y = mul(diag, v)
        y.index_add_(0, own, mul(upper, v[nei]))
        y.index_add_(0, nei, mul(lower, v[own]))
        return y

    x = mul(dinv, b)
    for _ in range(4):
        r = b - A(x)
        rw, p = r.clone(), r.clone()
        rho = (rw * r).sum()
        for _ in range(60):
            ph = mul(dinv, p)
            v = A(ph)
            alpha = rho / (rw * v).sum()
            q = r - alpha * v
            qh = mul(dinv, q)
            t = A(qh)
            tt = (t * t).sum()
            if float(tt) == 0.0:
                break
            om = (t * q).sum() / tt
            x = x + alpha * ph + om * qh
            r = q - om * t
            if float(r.norm()) < 1e-15 * float(b.norm()):
                break
            new = (rw * r).sum()
            p = r + (new / rho) * (alpha / om) * (p - om * v)
            rho = new
    return {"x": x.cpu()}
