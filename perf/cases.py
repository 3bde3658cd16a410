"""The work that users of this framework have it do, as measurable cases: resistance tensors of one
body and of a batch, boundary-value solves, integral assembly, post-processing of a flow, the dense
solvers and the training of the quadrature network.

listed() names the cases, draw() gives more of the same ranges, prepare() makes what a program holds
before the call, run() is the call, work() the bytes and flops it cannot do without and exact() the
same outputs in 64 bits without this framework, where they have such a value: the integrals by a
quadrature of high order, the linear systems by a direct solve. The tensors and boundary-value
solutions are those of the collocation scheme with its fixed triangle rule, so they have no value
apart from it (None).
"""
import math
import os

import numpy as np
import torch

from andromeda_amd import api
from andromeda_amd import mesh as M

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
RULE_POINTS = (0, 7, 25, 54, 85, 126)  # points of the triangle rules itri 1..5
MAX_BATCH_ELEMENTS = 110000            # a drawn batch is no larger than the listed one

_state = {}


def _context():
    """One context per process, with the shipped quadrature model, as a program keeps it."""
    if "ctx" not in _state:
        ctx = api.Context(0)
        z = np.load(os.path.join(ROOT, "andromeda_amd", "quad_model.npz"))
        ctx.set_quadrature_model(z["params"], float(z["confidence"]), float(z["near_ratio"]), z["far_table"])
        _state["ctx"] = ctx
    return _state["ctx"]


# ---- the cases ---------------------------------------------------------------------------------
def listed():
    return [
        # one small particle, the interactive call: launches and host time count
        {"name": "tensor_one_small", "kind": "tensor_fast", "body": "super", "nelem": 500, "form": "exterior",
         "precision": "mixed", "problems": "rigid"},
        # one ordinary slender particle in its far outer sphere, in the strain fields (Jeffery torques)
        {"name": "tensor_bounded_strain", "kind": "tensor_fast", "body": "fibre", "nelem": 2000, "form": "bounded",
         "precision": "mixed", "problems": "strain"},
        # the batched throughput job: resident bodies of 500 to 8000 elements, learned rule selection
        {"name": "tensor_batch_learned", "kind": "tensor_batch", "bodies": 40, "fibres": 4, "largest": 8000,
         "precision": "learned"},
        # the drop-in for the reference's particle run: FP64, bounded form, least squares
        {"name": "tensor_fp64_bounded", "kind": "tensor_fp64", "body": "super", "nelem": 720, "form": "bounded"},
        # heat conduction through nested spheres in contact, FP64, an ordinary model
        {"name": "laplace_contact", "kind": "laplace", "layers": 3, "nu": 6, "precision": "fp64", "quads": False},
        # one large single domain in the mixed form
        {"name": "laplace_mixed_large", "kind": "laplace", "layers": 1, "nu": 18, "precision": "mixed", "quads": False},
        # flow in a closed body, velocity on its lower wall and traction on the upper one
        {"name": "stokes_mixed_bc", "kind": "stokes", "nu": 6},
        # the integral matrices handed to a host solver
        {"name": "assemble_stokes", "kind": "assemble_stokes", "nelem": 720, "itri": 5, "pressure": True},
        # the same for the Laplace kernels on a quadrilateral mesh
        {"name": "assemble_laplace_quads", "kind": "assemble_laplace", "n": 10, "split": True, "iquad": 4, "itri": 5},
        # the field of a finished solve: domain points and surface pressure
        {"name": "flow_field", "kind": "flow_field", "nu_in": 5, "nu_out": 5, "npts": 1501, "itri": 5},
        # a dense system already on the device, several right-hand sides
        {"name": "bicgstab_device", "kind": "bicgstab", "n": 3841, "nrhs": 6},
        # an epoch of the quadrature network
        {"name": "mlp_train_epoch", "kind": "mlp", "n": 40000, "batch": 1024, "epochs": 1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tensor_fast", "tensor_fast", "tensor_batch", "tensor_fp64", "laplace", "stokes",
                       "assemble_stokes", "assemble_laplace", "flow_field", "bicgstab", "lsqr", "mlp"])
    c = {"kind": kind}
    if kind == "tensor_fast":
        c |= {"body": rng.choice(["super", "fibre"]), "nelem": _log(rng, 180, 8000),
              "form": rng.choice(["exterior", "bounded"]), "precision": rng.choice(["mixed", "learned"]),
              "problems": rng.choice(["rigid", "rigid", "strain"])}
    elif kind == "tensor_batch":
        largest = _log(rng, 1000, 8000)
        n = rng.randint(3, 40)
        c |= {"bodies": n, "fibres": rng.randint(0, max(1, n // 8)), "largest": largest,
              "precision": rng.choice(["mixed", "learned"])}
    elif kind == "tensor_fp64":
        c |= {"body": rng.choice(["super", "fibre"]), "nelem": _log(rng, 180, 1500),
              "form": rng.choice(["exterior", "bounded"])}
    elif kind == "laplace":
        layers, quads = rng.randint(1, 3), rng.random() < 0.3
        c |= {"layers": layers, "nu": _log(rng, 3, 18 if layers == 1 else 9), "precision": rng.choice(["fp64", "mixed"]),
              "quads": quads}
        if quads:  # a mesh of 6 nu^2 quadrilaterals per sphere, of about as many elements
            c["nu"] = min(c["nu"], 10)
    elif kind == "stokes":
        c |= {"nu": rng.randint(3, 9)}
    elif kind == "assemble_stokes":
        c |= {"nelem": _log(rng, 80, 1000), "itri": rng.choice([1, 3, 5, 5]), "pressure": rng.random() < 0.7}
    elif kind == "assemble_laplace":
        c |= {"n": rng.randint(3, 14), "split": rng.random() < 0.5, "iquad": rng.choice([2, 3, 4]),
              "itri": rng.choice([2, 4, 5])}
    elif kind == "flow_field":
        c |= {"nu_in": rng.randint(3, 8), "nu_out": rng.randint(2, 6), "npts": _log(rng, 20, 4000),
              "itri": rng.choice([3, 5, 5])}
    elif kind == "bicgstab":
        c |= {"n": _log(rng, 300, 9000), "nrhs": rng.choice([1, 2, 3, 6, 9])}
    elif kind == "lsqr":
        n = _log(rng, 200, 2500)
        c |= {"m": n + rng.randint(0, n // 2), "n": n, "nrhs": rng.choice([1, 3, 6])}
    else:
        c |= {"n": _log(rng, 3000, 60000), "batch": rng.choice([512, 1024, 4096]), "epochs": rng.choice([1, 1, 2])}
    return c


# ---- inputs ------------------------------------------------------------------------------------
def _body(rng, body, nelem):
    if body == "fibre":
        return M.random_fibre(rng, max(nelem, 180))[0]
    return M.random_superellipsoid(rng, max(3, int(round(math.sqrt(nelem / 20.0)))))[0]


def _outer_nu(nelem):
    """The far outer sphere of the bounded form is meshed coarser than the body."""
    return 3 if nelem < 500 else 4


def _formed(rng, case):
    """The body of a tensor case, in its outer sphere for the bounded form."""
    m = _body(rng, case["body"], case["nelem"])
    if case["form"] == "bounded":
        m = M.body_in_sphere(m, 12.0, _outer_nu(case["nelem"]))
    return m


def _form(case):
    return api.FORM_BOUNDED if case["form"] == "bounded" else api.FORM_EXTERIOR


def _batch_meshes(case, rng):
    """Element counts log-uniform in [500, largest], as the batched workload draws them."""
    meshes, total = [], 0
    for k in range(case["bodies"]):
        # the counts are those of the case, whatever the seed
        f = math.exp(math.log(500.0) + (math.log(case["largest"]) - math.log(500.0)) * ((k * 0.6180339887498949) % 1.0))
        total += f
        if total > MAX_BATCH_ELEMENTS and k > 2:
            break
        nu = M.nu_for_elements(f)
        if k >= case["bodies"] - case["fibres"]:
            meshes.append(M.random_fibre(rng, 20 * nu * nu)[0])
        else:
            meshes.append(M.random_superellipsoid(rng, nu)[0])
    return meshes


def _nested(case, scale):
    """Concentric spheres 1, 2, .. layers, each cut at its equator when it is the outermost: the outer
    sphere carries a known function on its lower half and a known flux on the upper one, the inner
    ones are contacts between subdomains of different diffusivity."""
    parts, walls = [], 0
    xyz, con, bcid, off = [], [], [], 0
    L = case["layers"]
    for k in range(1, L + 1):
        s = M.cubed_sphere(case["nu"], scale * k) if case["quads"] else M.geodesic_sphere(case["nu"], scale * k)
        z = s.xyz[s.con].mean(axis=1)[:, 2]
        xyz.append(s.xyz)
        con.append(s.con + off)
        bcid.append(np.where(z < 0.0, walls + 1, walls + 2) if k == L else np.full(s.nelem, walls + 1))
        parts.append([walls + 1, walls + 2] if k == L else [walls + 1])
        walls += len(parts[-1])
        off += s.nnodes
    mesh = M.Mesh(np.vstack(xyz), np.vstack(con).astype(np.int32), np.concatenate(bcid).astype(np.int32), "nested")
    sds = []
    for k in range(L):  # subdomain k lies between sphere k (normals turned inwards) and sphere k + 1
        inner = parts[k - 1] if k else []
        sds.append(api.Subdomain(parts[k] + inner, [1.0] * len(parts[k]) + [-1.0] * len(inner), 1.0 + 0.5 * k))
    bc = [api.BC_CONTACT] * (walls - 2) + [api.BC_FUNCTION, api.BC_FLUX]
    return mesh, sds, np.array([bc], dtype=np.int32)


def _stokeslet(x, n, x0, f):
    """Velocity and traction (normal n) at x of a point force f at x0, viscosity 1."""
    r = x - x0
    d = np.linalg.norm(r, axis=1)[:, None]
    rf = (r * f).sum(axis=1)[:, None]
    u = (f / d + r * rf / d ** 3) / (8 * math.pi)
    t = -3.0 / (4 * math.pi) * r * rf * (r * n).sum(axis=1)[:, None] / d ** 5
    return u, t


def _geometry(m):
    a, b, c = (m.xyz[m.con[:, k]] for k in range(3))
    n = np.cross(b - a, c - a)
    d = np.linalg.norm(n, axis=1)[:, None]
    return n / d, 0.5 * d[:, 0], (a + b + c) / 3.0


def _flow_mesh(case, rng):
    body = M.random_superellipsoid(rng, case["nu_in"])[0]
    return M.body_in_sphere(body, 6.0, case["nu_out"])


def _records(rng, n):
    """Pair records of the training set: distance, aspect, normal angle, kernel; the label grows as the
    pair gets nearer, more distorted, more oblique."""
    d = np.exp(rng.uniform(math.log(0.4), math.log(4.0), n))
    a = np.exp(np.abs(rng.normal(0.15, 0.25, n)))
    c = rng.uniform(-1.0, 1.0, n)
    k = rng.integers(0, 3, n)
    f = np.zeros((n, 6), dtype=np.float32)
    f[:, 0], f[:, 1], f[:, 2] = np.log(d), np.log(a), c
    f[np.arange(n), 3 + k] = 1.0
    s = 5.2 - 3.1 * np.log(d) + 1.1 * np.log(a) + 0.4 * k + 0.3 * c + rng.normal(0.0, 0.15, n)
    return f, np.clip(np.round(s), 0, 7).astype(np.int32)


def _kernel_system(n, nrhs, seed):
    """The single-layer collocation system of a wavy sphere, on the device: the weighted 1 / r kernel
    with the self-integral of a disc of the same area on the diagonal, and right-hand sides of smooth
    fields with some noise."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    i = torch.arange(n, device="cuda", dtype=torch.float64) + 0.5
    z = 1.0 - 2.0 * i / n
    phi = math.pi * (1.0 + math.sqrt(5.0)) * i
    w = torch.randn(8, generator=g, device="cuda", dtype=torch.float64)
    s = torch.sqrt(1.0 - z * z)
    x = torch.stack([s * torch.cos(phi), s * torch.sin(phi), z], 1)
    rad = 1.0 + 0.05 * (w[0] * torch.sin(3 * phi) * s ** 3 + w[1] * z * z + w[2] * x[:, 0] * z)
    x = x * rad[:, None]
    A = torch.zeros(n, n, dtype=torch.float64, device="cuda")
    for k in range(3):
        A += (x[:, None, k] - x[None, :, k]) ** 2
    A.fill_diagonal_(1.0)
    A.rsqrt_()
    A *= 1.0 / n
    A.fill_diagonal_(1.0 / math.sqrt(n))
    c = torch.randn(nrhs, 4, generator=g, device="cuda", dtype=torch.float64)
    B = (c[:, :3] @ x.T + c[:, 3:] * (x[:, 0] * x[:, 1])[None] +
         0.05 * torch.randn(nrhs, n, generator=g, device="cuda", dtype=torch.float64)).contiguous()
    return A.contiguous(), B


def _ls_system(case, rng):
    """A well-posed overdetermined system: identity and random coupling, columns of different scale."""
    m, n = case["m"], case["n"]
    A = rng.standard_normal((m, n)) * (0.4 / math.sqrt(m))
    A[np.arange(n), np.arange(n)] += 1.0
    A *= np.exp(rng.uniform(-1.0, 1.0, n))[None, :]
    return A, rng.standard_normal((m, case["nrhs"]))


def prepare(case, seed):
    kind, rng = case["kind"], np.random.default_rng(seed)
    s = {"kind": kind, "case": case, "ctx": _context()}
    if kind in ("tensor_fast", "tensor_fp64"):
        s["mesh"] = _formed(rng, case)
    elif kind == "tensor_batch":
        s["bodies"] = s["ctx"].upload_bodies(_batch_meshes(case, rng))
    elif kind == "laplace":
        scale = float(rng.uniform(0.5, 2.0))
        mesh, sds, bc = _nested(case, scale)
        c = rng.normal(size=4)
        x = mesh.xyz / scale
        u = c[0] + x @ c[1:] + 0.5 * x[:, 0] * x[:, 1]
        q = rng.normal() + mesh.xyz[mesh.con].mean(axis=1)[:, 0] / scale
        outer = mesh.bcid >= mesh.nwalls - 1
        u_known = np.zeros(mesh.nnodes, dtype=bool)
        u_known[np.unique(mesh.con[outer])] = True
        s |= {"mesh": mesh, "sds": sds, "bc": bc, "u": np.where(u_known, u, 0.0)[None],
              "q": np.where(mesh.bcid == mesh.nwalls, q, 0.0)[None]}
    elif kind == "stokes":
        mesh = M.random_superellipsoid(rng, case["nu"])[0]
        n, _, cen = _geometry(mesh)
        mesh.bcid = np.where(cen[:, 2] > 0.0, 2, 1).astype(np.int32)
        f, x0 = rng.normal(size=3), np.array([0.0, 0.0, -6.0])
        u, _ = _stokeslet(mesh.xyz, mesh.xyz, x0, f)
        _, t = _stokeslet(cen, n, x0, f)
        known = np.unique(mesh.con[mesh.bcid == 1])
        u[np.setdiff1d(np.arange(mesh.nnodes), known)] = 0.0
        t[mesh.bcid == 1] = 0.0
        s |= {"mesh": mesh, "sd": api.Subdomain([2, 1]), "u": u.T.copy(), "q": -t.T.copy(),
              "bc": np.array([[api.BC_FUNCTION, api.BC_FLUX]] * 3, dtype=np.int32)}
    elif kind == "assemble_stokes":
        s["mesh"] = _body(rng, "super", case["nelem"])
    elif kind == "assemble_laplace":
        mesh = M.cubed_sphere(case["n"])
        mesh.xyz = mesh.xyz * rng.uniform(0.5, 2.0, 3)[None]
        s["mesh"] = M.split_some_quads(mesh) if case["split"] else mesh
    elif kind == "flow_field":
        mesh = _flow_mesh(case, rng)
        n, _, cen = _geometry(mesh)
        f, x0 = rng.normal(size=3), rng.uniform(-0.1, 0.1, 3)
        u, _ = _stokeslet(mesh.xyz, mesh.xyz, x0, f)
        _, t = _stokeslet(cen, n, x0, f)
        d = rng.normal(size=(case["npts"], 3))
        s |= {"mesh": mesh, "u": u, "q": t,
              "pts": d / np.linalg.norm(d, axis=1)[:, None] * rng.uniform(3.2, 4.4, (case["npts"], 1))}
    elif kind == "bicgstab":
        A, B = _kernel_system(case["n"], case["nrhs"], seed)
        s |= {"A": A, "B": B, "X": torch.zeros_like(B)}
        torch.cuda.synchronize()
    elif kind == "lsqr":
        s["A"], s["B"] = _ls_system(case, rng)
    else:
        s["f"], s["l"] = _records(rng, case["n"])
        w = [rng.standard_normal(a * b) * math.sqrt(2.0 / a) for a, b in ((6, 64), (64, 64), (64, 64), (64, 8))]
        s["p"] = np.concatenate([v for k, b in zip(w, (64, 64, 64, 8)) for v in (k, np.zeros(b))]).astype(np.float32)
    return s


# ---- the calls ---------------------------------------------------------------------------------
_PREC = {"fp64": api.PREC_FP64, "mixed": api.PREC_MIXED, "learned": api.PREC_LEARNED}


def run(s):
    """The calls' results. The self-check errors that some calls also report are left out: they are
    rounding noise around zero, and so are the iteration counts and times."""
    kind, case, ctx = s["kind"], s["case"], s["ctx"]
    if kind == "tensor_fast":
        problems = api.PROBLEMS_STRAIN if case["problems"] == "strain" else api.PROBLEMS_RIGID
        return ctx.resistance(s["mesh"], form=_form(case), precision=_PREC[case["precision"]], problems=problems).FT
    if kind == "tensor_fp64":
        return ctx.resistance(s["mesh"], form=_form(case), precision=api.PREC_FP64).FT
    if kind == "tensor_batch":
        return np.stack([r.FT for r in ctx.resistance_batch_resident(s["bodies"], precision=_PREC[case["precision"]])])
    if kind == "laplace":
        r = ctx.laplace_solve(s["mesh"], s["sds"], s["bc"], s["u"], s["q"], eps=1e-13, maxit=0,
                              precision=_PREC[case["precision"]])[0]
        return {"u": r.u, "q": r.q, "flux": r.wall_flux}
    if kind == "stokes":
        r = ctx.stokes_solve(s["mesh"], s["sd"], s["bc"], s["u"], s["q"], eps=1e-13, maxit=0)
        return {"u": r.u, "q": r.q, "force": r.wall_flux}
    if kind == "assemble_stokes":
        T, G, pT, pG, _ = ctx.assemble_stokes(s["mesh"], itri=case["itri"], pressure=case["pressure"])
        return {"T": T, "G": G, "prT": pT or [], "prG": pG or []}
    if kind == "assemble_laplace":
        H, G, _ = ctx.assemble_laplace(s["mesh"], itri=case["itri"], iquad=case["iquad"])
        return {"H": H, "G": G}
    if kind == "flow_field":
        v, p, _ = ctx.stokes_domain_values(s["mesh"], s["pts"], s["u"], s["q"], itri=case["itri"])
        return {"velocity": v, "pressure": p,
                "surface": ctx.stokes_surface_pressure(s["mesh"], s["u"], s["q"], itri=case["itri"])}
    if kind == "bicgstab":
        n = case["n"]
        s["X"].zero_()
        torch.cuda.current_stream().synchronize()  # the context works on a stream of its own
        ctx.bicgstab_dense_noalloc(n, s["A"].data_ptr(), n, case["nrhs"], s["B"].data_ptr(), s["X"].data_ptr(),
                                   tol=1e-10)
        return s["X"]
    if kind == "lsqr":
        return ctx.lsqr_dense(s["A"], s["B"], eps=1e-12)[0]
    p, loss = ctx.mlp_train(s["f"], s["l"], s["p"], epochs=case["epochs"], batch=case["batch"], seed=3)
    return {"params": p, "loss": loss}


# ---- what a pass cannot do without ---------------------------------------------------------------
def _counts(case):
    """(elements, nodes) of a case's mesh."""
    kind = case["kind"]
    if kind in ("tensor_fast", "tensor_fp64"):
        e = case["nelem"]
        if case["form"] == "bounded":
            e += 20 * _outer_nu(case["nelem"]) ** 2
        return e, e // 2 + 2
    if kind == "stokes":
        return 20 * case["nu"] ** 2, 10 * case["nu"] ** 2 + 2
    if kind == "flow_field":
        e = 20 * (case["nu_in"] ** 2 + case["nu_out"] ** 2)
        return e, e // 2 + 4
    if kind == "laplace":
        e = case["layers"] * (6 if case["quads"] else 20) * case["nu"] ** 2
        return e, e + 2 if case["quads"] else e // 2 + 2
    if kind == "assemble_laplace":
        e = 6 * case["n"] ** 2
        return (e * 4) // 3 if case["split"] else e, e + 2
    return case["nelem"], case["nelem"] // 2 + 2


def work(case):
    """Flops: 107 per quadrature point of a Stokes pair, 60 where only vertex sums are needed, 50 of a
    Laplace pair, plus the products of the iterative solves at the iteration counts these systems
    take. Bytes: the inputs and results of a call, plus the system read once per product, as no
    product can start before the one ahead of it."""
    kind = case["kind"]
    if kind == "bicgstab":
        n, r = case["n"], case["nrhs"]
        its = 36 * -(-r // 8)
        return {"bytes": 2 * its * 8.0 * n * n, "flops": 2 * its * 2.0 * n * n * min(r, 8)}
    if kind == "lsqr":
        m, n, r = case["m"], case["n"], case["nrhs"]
        return {"bytes": 35 * 2 * 8.0 * m * n, "flops": 35 * 4.0 * m * n * r}
    if kind == "mlp":
        n = case["n"] * case["epochs"]
        return {"bytes": 4.0 * 7 * n + 8 * 9288.0, "flops": 3 * 2.0 * 9088 * n}
    if kind == "tensor_batch":
        b = f = total = 0.0
        for k in range(case["bodies"]):
            e = math.exp(math.log(500.0) + (math.log(case["largest"]) - math.log(500.0)) * ((k * 0.6180339887498949) % 1.0))
            total += e
            if total > MAX_BATCH_ELEMENTS and k > 2:
                break
            points = 7 if case["precision"] == "learned" else 126
            b += 20 * 24.0 * e * e
            f += 60.0 * points * e * e + 20 * 2.0 * 9 * e * e * 6
        return {"bytes": b, "flops": f}
    e, v = _counts(case)
    if kind == "tensor_fast":
        points = 7 if case["precision"] == "learned" else 126
        its = 70 if case["body"] == "fibre" else 20
        return {"bytes": its * 24.0 * e * e, "flops": 60.0 * points * e * e + its * 2.0 * 9 * e * e * 6}
    if kind == "tensor_fp64":
        its = 1200 if case["body"] == "fibre" else 300
        return {"bytes": its * 2 * 72.0 * e * e, "flops": 107.0 * 126 * e * e + its * 4.0 * 9 * e * e * 6}
    if kind == "laplace":
        its, rows, n = (300, 0.75 * e, 0.75 * e) if case["layers"] == 1 else (400, 2.2 * e, 1.25 * e)
        per = 8.0 if case["precision"] == "fp64" else 4.0
        evals = case["layers"] * (2 * e / case["layers"]) * (1.5 * e / case["layers"]) * (256 if case["quads"] else 126)
        return {"bytes": its * 2 * per * rows * n, "flops": 50.0 * evals + its * 4.0 * rows * n}
    if kind == "stokes":
        n, its = 3 * 0.75 * e, 200
        return {"bytes": its * 2 * 8.0 * n * n, "flops": 107.0 * 126 * 1.5 * e * e + its * 4.0 * n * n}
    points = RULE_POINTS[case["itri"]]
    if kind == "assemble_stokes":
        k = 9 if case["pressure"] else 6
        return {"bytes": 8.0 * k * (e + v) * (e + v), "flops": 107.0 * points * (e + v) * e}
    if kind == "assemble_laplace":
        points = 4 * (0, 2, 4, 6, 8)[case["iquad"]] ** 2
        return {"bytes": 8.0 * (e + v) * (e + v), "flops": 50.0 * points * (e + v) * e}
    evals = points * e * float(case["npts"] + e)
    return {"bytes": 8.0 * (7 * case["npts"] + 6 * v + 8 * e), "flops": 60.0 * evals}


# ---- the same outputs in 64 bits -----------------------------------------------------------------
def _square_rule(k):
    """Triangle rule in barycentric coordinates: Gauss points of the square folded onto the first corner,
    which also takes a 1 / r singularity in that corner."""
    g, w = np.polynomial.legendre.leggauss(k)
    g, w = 0.5 * (g + 1.0), 0.5 * w
    t, s = np.meshgrid(g, g, indexing="ij")
    wt = (np.outer(w, w) * t * 2.0).ravel()  # weights sum to 1
    t, s = t.ravel(), s.ravel()
    return np.stack([1.0 - t, t * (1.0 - s), t * s], 1), wt


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _tri_points(m, bary):
    """Points (elements, quadrature, 3) of a rule on every triangle."""
    return torch.einsum("qv,evd->eqd", _dev(bary), _dev(m.xyz[m.con]))


OSEM = 8.0 * 4.0 * float(np.arctan(np.float32(1.0)))  # 8 pi as the scheme holds it


def _exact_flow(s):
    m = s["mesh"]
    n, area, cen = _geometry(m)
    bary, w = _square_rule(16)
    n, area, W, L = _dev(n), _dev(area), _dev(w), _dev(bary)
    Y = _tri_points(m, bary)
    U = torch.einsum("qv,evd->eqd", L, _dev(s["u"][m.con]))
    Q = _dev(s["q"])
    jac = area[:, None] * W[None]

    def at(p, skip=None):
        r = Y - p
        i2 = 1.0 / (r * r).sum(-1)
        i1 = torch.sqrt(i2)
        rn, ru = (r * n[:, None]).sum(-1), (r * U).sum(-1)
        rq, un = (r * Q[:, None]).sum(-1), (U * n[:, None]).sum(-1)
        j = jac if skip is None else jac * (torch.arange(jac.shape[0], device="cuda") != skip)[:, None]
        vel = (j * -6.0 * rn * ru * i1 * i2 * i2)[..., None] * r + (j * i1)[..., None] * Q[:, None] + (j * rq * i1 * i2)[..., None] * r
        pu = j * 4.0 * i1 * i2 * (3.0 * rn * ru * i2 - un)
        pq = j * 2.0 * rq * i1 * i2
        one = (j * 4.0 * i1 * i2)[..., None] * (3.0 * (rn * i2)[..., None] * r - n[:, None])  # row sums of prT
        return vel.sum((0, 1)), pu.sum(), pq.sum(), one.sum((0, 1))

    V, P, S = [], [], []
    for p in _dev(s["pts"]):
        v, pu, pq, _ = at(p)
        V.append(-v / OSEM)
        P.append(-(pu - pq) / OSEM)
    uc = _dev(s["u"][m.con].mean(axis=1))
    for e, p in enumerate(_dev(cen)):
        _, pu, pq, one = at(p, e)
        S.append(-2.0 * (pu - (one * uc[e]).sum() - pq) / OSEM)
    return {"velocity": torch.stack(V), "pressure": torch.stack(P), "surface": torch.stack(S)}


_SYM = ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))


def _exact_stokes(case, m):
    """The integral matrices row by row; a singular pair (the source on the element) has a Stokeslet
    integral only, taken over the triangles that meet in the source."""
    n, area, cen = _geometry(m)
    con, nn, ne = _dev(m.con.astype(np.int64)), m.nnodes, m.nelem
    N, A = _dev(n), _dev(area)
    bary, w = _square_rule(12)
    W, L, Y = _dev(w), _dev(bary), _tri_points(m, bary)
    src = _dev(np.vstack([m.xyz, cen]))
    nsp = nn + ne
    T = torch.zeros(6, nsp, nn, dtype=torch.float64, device="cuda")
    G = torch.zeros(6, nsp, ne, dtype=torch.float64, device="cuda")
    pT = torch.zeros(3, nsp, nn, dtype=torch.float64, device="cuda")
    pG = torch.zeros(3, nsp, ne, dtype=torch.float64, device="cuda")
    fine, fw = _square_rule(24)
    fine, fw = _dev(fine), _dev(fw)
    touching = [[] for _ in range(nn)]
    for e, c in enumerate(m.con):
        for v in c:
            touching[v].append(e)
    x = _dev(m.xyz)

    def stokeslet(p, corners, a):  # corners (k, 3, 3), the first one the source
        r = torch.einsum("qv,kvd->kqd", fine, corners) - p
        d = torch.sqrt((r * r).sum(-1))
        return [((a[:, None] * fw[None]) * ((1.0 if i == j else 0.0) / d + r[..., i] * r[..., j] / d ** 3)).sum(1) for i, j in _SYM]

    for k in range(nsp):
        p = src[k]
        own = torch.tensor(touching[k] if k < nn else [k - nn], device="cuda")
        r = Y - p
        i2 = 1.0 / (r * r).sum(-1)
        i1 = torch.sqrt(i2)
        jac = A[:, None] * W[None]
        jac[own] = 0.0
        rn = (r * N[:, None]).sum(-1)
        for c, (i, j) in enumerate(_SYM):
            rr = r[..., i] * r[..., j]
            G[c, k] = (jac * i1 * ((1.0 if i == j else 0.0) + rr * i2)).sum(1)
            t = (jac * -6.0 * rn * rr * i1 * i2 * i2) @ L
            T[c, k].index_add_(0, con.reshape(-1), t.reshape(-1))
        for i in range(3):
            pG[i, k] = (jac * 2.0 * r[..., i] * i1 * i2).sum(1)
            t = (jac * 4.0 * i1 * i2 * (3.0 * rn * r[..., i] * i2 - N[:, None, i])) @ L
            pT[i, k].index_add_(0, con.reshape(-1), t.reshape(-1))
        if k < nn:
            c = con[own]
            first = (c == k).to(torch.int64).argmax(1)
            order = (first[:, None] + torch.arange(3, device="cuda")) % 3
            g = stokeslet(p, x[c.gather(1, order)], A[own])
            for q in range(6):
                G[q, k, own] = g[q]
            for q in (0, 3, 5):
                T[q, k, k] -= T[q, k].sum()
        else:
            e = k - nn
            v = x[con[e]]
            corners = torch.stack([torch.stack([p, v[j], v[(j + 1) % 3]]) for j in range(3)])
            a = 0.5 * torch.linalg.norm(torch.linalg.cross(corners[:, 1] - p, corners[:, 2] - p), dim=1)
            for q, g in enumerate(stokeslet(p, corners, a)):
                G[q, k, e] = g.sum()
            for q in (0, 3, 5):
                T[q, k, con[e]] -= T[q, k].sum() / 3.0
            for q in range(3):
                pT[q, k, con[e]] -= pT[q, k].sum() / 3.0
    press = case["pressure"]
    return {"T": list(T), "G": list(G), "prT": list(pT) if press else [], "prG": list(pG) if press else []}


def exact(case, seed):
    kind = case["kind"]
    if kind == "flow_field":
        return _exact_flow(prepare(case, seed)) if case["npts"] + _counts(case)[0] < 5000 else None
    if kind == "assemble_stokes":
        return _exact_stokes(case, prepare(case, seed)["mesh"])
    if kind == "bicgstab":
        A, B = _kernel_system(case["n"], case["nrhs"], seed)
        return torch.linalg.solve(A, B.T).T
    if kind == "lsqr":
        A, B = _ls_system(case, np.random.default_rng(seed))
        q, r = torch.linalg.qr(_dev(A))
        return torch.linalg.solve_triangular(r, q.T.contiguous() @ _dev(B), upper=True)
    return None
