"""The work that users of this framework have it do, as cases that can be
timed: explicit central-difference runs through the public entry points
(``SolidMechanicsModel``, ``Batch``, ``serving.Server``).

Every case is a jittered box of _tetrahedron_4 (6 per cell) or _hexahedron_8
elements, clamped at x = 0 and started with a random velocity field, as in
bench.py and the tests.  One pass advances the simulation by a number of steps
and reads back displacement, velocity and internal force, as a program does
between two outputs.  Sizes run from the 1,920-element bar of the parity tests
to the 2 million Hex8 of the benchmark and the 4.4 million Tet4 of the
published scaling study; single models, batches and served requests; FP64 and
the FP32 form; all four built-in laws.

The FP32 form's fields are handed on in float32, the precision its forces have
(a dump of them holds no more); those of FP64 runs stay float64.
"""
import math

import numpy as np
import torch

from akantu2_amd import SolidMechanicsModel
from akantu2_amd import serving
from akantu2_amd.batch import Batch
from akantu2_amd.mesh import BoxMesh

TET4, HEX8 = "tet4", "hex8"
ELASTIC, ELASTIC_FD, NEO = "elastic", "elastic_fd", "neohookean"
PLASTIC = "plastic_linear_isotropic_hardening"
LAWS = (ELASTIC, ELASTIC_FD, NEO, PLASTIC)
FIELDS = ("displacement", "velocity", "internal_force")


def _model(name, etype, cells, law, precision, steps, per_element=False, loop=False):
    return dict(name=name, kind="model", etype=etype, nx=cells[0], ny=cells[1], nz=cells[2],
                law=law, precision=precision, steps=steps, per_element=per_element, loop=loop)


def _many(name, kind, etype, law, precision, steps, count, smallest, largest):
    return dict(name=name, kind=kind, etype=etype, law=law, precision=precision, steps=steps,
                count=count, smallest=smallest, largest=largest)


def listed():
    return [
        # the smallest user program: a small bar stepped by a solveStep() loop
        _model("bar tet4 elastic, step loop", TET4, (20, 4, 4), ELASTIC, "fp64", 100, loop=True),
        # small boxes, many steps in one call: launches and latency count
        _model("hex8 1e3 neo-Hookean", HEX8, (10, 10, 10), NEO, "fp64", 300),
        _model("tet4 5e3 elastic f32", TET4, (17, 7, 7), ELASTIC, "fp32", 300),
        # ordinary sizes
        _model("tet4 35e3 plastic", TET4, (30, 14, 14), PLASTIC, "fp64", 200),
        _model("hex8 20e3 neo-Hookean f32", HEX8, (47, 21, 20), NEO, "fp32", 300),
        # the benchmark's box, plain FP64 and in the FP32 form
        _model("hex8 2e6 neo-Hookean", HEX8, (200, 100, 100), NEO, "fp64", 100),
        _model("hex8 2e6 neo-Hookean f32", HEX8, (200, 100, 100), NEO, "fp32", 200),
        # a heterogeneous body, E and nu of its own in every element
        _model("tet4 1.9e6 elastic E(x) f32", TET4, (131, 49, 49), ELASTIC, "fp32", 300,
               per_element=True),
        # the published scaling study: 4.4 million Tet4, finite strain
        _model("tet4 4.4e6 finite strain", TET4, (90, 90, 90), ELASTIC_FD, "fp64", 100),
        # parameter studies: many boxes of uneven size stepped together
        _many("batch tet4 plastic f32", "batch", TET4, PLASTIC, "fp32", 200, 20, 5000, 200000),
        _many("batch hex8 neo-Hookean", "batch", HEX8, NEO, "fp64", 100, 12, 1000, 60000),
        # requests of both element types that wait for the server together
        _many("serve f32", "serve", "both", "both", "fp32", 250, 12, 1000, 100000),
    ]


def draw(rng):
    """One more case of the same ranges.  The steps of a pass are fewer the
    larger the mesh, so that no drawn case costs more than the largest."""
    def logu(a, b):
        return math.exp(rng.uniform(math.log(a), math.log(b)))
    kind = rng.choice(("model", "model", "model", "model", "batch", "serve"))
    precision = rng.choice(("fp64", "fp32"))
    etype = rng.choice((TET4, HEX8))
    if kind == "model":
        # the FP32 form of the single model keeps the plastic law's full
        # incremental history, so plasticity is run in FP64 or in batches
        law = rng.choice(LAWS if precision == "fp64" else LAWS[:3])
        most = 4e6 if etype == TET4 else 2e6
        if law == PLASTIC:
            most = 3e5
        cells = _cells(etype, logu(1e3, most), rng.uniform(1.0, 8.0), rng)
        nel = cells[0] * cells[1] * cells[2] * (6 if etype == TET4 else 1)
        loop = nel < 2e4 and rng.random() < 0.4
        steps = 100 if loop else max(20, min(300, int(6e7 / nel)))
        per_element = law in (ELASTIC, ELASTIC_FD) and rng.random() < 0.4
        c = _model("", etype, cells, law, precision, steps, per_element, loop)
    elif kind == "batch":
        law = rng.choice(LAWS if etype == TET4 else LAWS[:3])
        most = logu(2e4, 2e5) if etype == TET4 else logu(5e3, 6e4)
        c = _many("", "batch", etype, law, precision, 100, rng.randint(3, 20), 1000, int(most))
    else:
        c = _many("", "serve", "both", "both", precision, 200, rng.randint(3, 12), 1000,
                  int(logu(1e4, 1e5)))
    del c["name"]
    return c


def _cells(etype, nel, aspect, rng):
    n = nel / (6 if etype == TET4 else 1)
    ny = max(2, round((n / aspect) ** (1.0 / 3.0)))
    nz = max(2, ny + rng.choice((-1, 0, 0, 1)))
    return max(2, round(n / (ny * nz))), ny, nz


# --------------------------------------------------------------------------
# inputs: meshes, materials, initial fields
# --------------------------------------------------------------------------
_CUBE = np.array([0, 1, 3, 2, 4, 5, 7, 6])  # corner bits (x, y, z) of Hex8 nodes 0..7
# six tetrahedra along the cube's diagonal, det J > 0 with xi -> node 3,
# eta -> node 1, zeta -> node 2
_KUHN = np.array([[0, 1, 3, 7], [0, 5, 1, 7], [0, 3, 2, 7], [0, 2, 6, 7],
                  [0, 4, 5, 7], [0, 6, 4, 7]])


def _box(etype, nx, ny, nz, seed):
    """Nodes [nn][3] and connectivity of a unit-cell box, x fastest, interior
    nodes moved by U(-0.1, 0.1); the clamped x = 0 face; the velocity envelope."""
    rng = np.random.default_rng(seed)
    shape = (nz + 1, ny + 1, nx + 1)
    nodes = np.empty(shape + (3,))
    nodes[..., 0] = np.arange(nx + 1)
    nodes[..., 1] = np.arange(ny + 1)[:, None]
    nodes[..., 2] = np.arange(nz + 1)[:, None, None]
    nodes[1:-1, 1:-1, 1:-1] += rng.uniform(-0.1, 0.1, (nz - 1, ny - 1, nx - 1, 3))
    first = np.arange(shape[0] * shape[1] * shape[2], dtype=np.int32).reshape(shape)
    first = first[:-1, :-1, :-1].reshape(-1)
    sx, sxy = nx + 1, (nx + 1) * (ny + 1)
    step = np.array([(b & 1) + sx * ((b >> 1) & 1) + sxy * (b >> 2) for b in range(8)], np.int32)
    if etype == HEX8:
        conn = first[:, None] + step[_CUBE]
    else:
        conn = (first[:, None, None] + step[_KUHN]).reshape(-1, 4)
    nodes = nodes.reshape(-1, 3)
    return nodes, np.ascontiguousarray(conn, np.int32), rng


def _inputs(etype, cells, law, seed, per_element=False):
    nodes, conn, rng = _box(etype, *cells, seed)
    blocked = np.zeros((nodes.shape[0], 3), np.uint8)
    blocked[nodes[:, 0] == 0.0] = 1
    amplitude = 1e-2 if law == PLASTIC else 1e-3
    v = amplitude * np.sin(np.pi * nodes[:, :1] / cells[0]) * rng.uniform(-1, 1, nodes.shape)
    mat = dict(rho=1.0, E=float(rng.uniform(0.5, 2.0)), nu=float(rng.uniform(0.2, 0.35)))
    if law == PLASTIC:
        mat.update(sigma_y=float(rng.uniform(1e-3, 5e-3)), h=float(rng.uniform(0.0, 0.1)))
    if per_element:
        mat["E_el"] = np.exp(rng.uniform(np.log(0.5), np.log(2.0), conn.shape[0]))
        mat["nu_el"] = rng.uniform(0.2, 0.35, conn.shape[0])
    mesh = BoxMesh(0 if etype == TET4 else 1, nodes, conn, tuple(cells))
    return dict(mesh=mesh, law=law, blocked=blocked, velocity=v, mat=mat, etype=etype)


def _instances(case, seed):
    """The instances of a batch or a server's queue: sizes spread over the
    logarithm of the range, the smallest and the largest among them."""
    rng = np.random.default_rng([seed, 7])
    out = []
    for k in range(case["count"]):
        t = k / max(1, case["count"] - 1)
        nel = case["smallest"] * (case["largest"] / case["smallest"]) ** t
        etype = case["etype"] if case["etype"] != "both" else (TET4, HEX8)[k % 2]
        law = case["law"] if case["law"] != "both" else (ELASTIC, NEO)[(k // 2) % 2]
        n = nel / (6 if etype == TET4 else 1)
        ny = max(2, int(round((n / (1.0 + 5.0 * ((0.38 * k) % 1.0))) ** (1.0 / 3.0))))
        cells = (max(2, int(round(n / (ny * ny)))), ny, ny)
        out.append(_inputs(etype, cells, law, int(rng.integers(1 << 30))))
    return out


def prepare(case, seed):
    if case["kind"] == "model":
        cells = (case["nx"], case["ny"], case["nz"])
        p = _inputs(case["etype"], cells, case["law"], seed, case["per_element"])
        m = SolidMechanicsModel(p["mesh"])
        m.addMaterial(p["law"], **p["mat"])
        m.setPrecision(case["precision"])
        m.initFull()
        m.getBlockedDOFs()[:] = p["blocked"]
        m.getVelocity()[:] = p["velocity"]
        m.setTimeStep(0.5 * m.getStableTimeStep())
        return dict(case=case, model=m)
    inst = _instances(case, seed)
    if case["kind"] == "batch":
        tets = sum(p["mesh"].nb_elements for p in inst if p["etype"] == TET4)
        hexes = sum(p["mesh"].nb_elements for p in inst if p["etype"] == HEX8)
        b = Batch(case["precision"], nodes=sum(p["mesh"].nb_nodes + 255 for p in inst),
                  tets=tets, hexes=hexes, plastic=case["law"] == PLASTIC)
        ids = [b.add(p["mesh"], p["law"], blocked=p["blocked"], velocity=p["velocity"],
                     dt_factor=0.5, **p["mat"]) for p in inst]
        return dict(case=case, batch=b, ids=ids)
    return dict(case=case, server=serving.Server(case["precision"], hbm_bytes=1 << 30),
                inputs=inst)


def _out(x, case):
    """A field as the program keeps it."""
    t = torch.from_numpy(np.asarray(x))
    return t.to(torch.float32) if case["precision"] == "fp32" else t


def run(state):
    case = state["case"]
    if case["kind"] == "model":
        m = state["model"]
        if case["loop"]:
            for _ in range(case["steps"]):
                m.solveStep()
        else:
            m.solveSteps(case["steps"])
        return [_out(m.getDisplacement(), case), _out(m.getVelocity(), case),
                _out(m.getInternalForce(), case)]
    if case["kind"] == "batch":
        b = state["batch"]
        b.solveStep(case["steps"])
        return [[_out(b.get(i, f), case) for f in FIELDS] for i in state["ids"]]
    requests = [serving.Request(k, 0.0, p["etype"], p["mesh"].shape, p["law"], p["mat"],
                                case["steps"] + 3 * k, 0, mesh=p["mesh"], blocked=p["blocked"],
                                velocity=p["velocity"])
                for k, p in enumerate(state["inputs"])]
    state["server"].run(requests)
    return [[_out(r.result[f], case) for f in FIELDS] for r in requests]


# --------------------------------------------------------------------------
# what one pass cannot do without
# --------------------------------------------------------------------------
# floating-point operations per Gauss point: the gradient, the law and the
# nodal forces, J^-1 and dN/dX taken as given
_LAW_FLOPS = {ELASTIC: 30, ELASTIC_FD: 130, NEO: 165, PLASTIC: 100}


def _work(etype, nn, nel, law, precision, steps, per_element=False):
    nnpe, nqp = (4, 1) if etype == TET4 else (8, 8)
    f32 = precision == "fp32"
    # per step: connectivity; X, mass, blocked bits; u and v read and written
    # (and a in FP64, compensation terms in FP32); element constants; history
    node = 24 + 8 + 1 + 2 * 24 * 2 + (2 * 24 if f32 else 2 * 24)
    elem = 4 * nnpe + ((8 if f32 else 16) if per_element else 0)
    if law == PLASTIC:
        elem += nqp * 2 * 7 * (4 if f32 else 8)
    flops = nel * nqp * (2 * 2 * 9 * nnpe + _LAW_FLOPS[law]) + nn * 30
    return (steps * (nn * node + nel * elem) + 3 * nn * (12 if f32 else 24), steps * flops)


def work(case):
    if case["kind"] == "model":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        nel = nx * ny * nz * (6 if case["etype"] == TET4 else 1)
        parts = [_work(case["etype"], (nx + 1) * (ny + 1) * (nz + 1), nel, case["law"],
                       case["precision"], case["steps"], case["per_element"])]
    else:
        parts = [_work(p["etype"], p["mesh"].nb_nodes, p["mesh"].nb_elements, p["law"],
                       case["precision"],
                       case["steps"] + (3 * k if case["kind"] == "serve" else 0))
                 for k, p in enumerate(_instances(case, 1))]
    return {"bytes": float(sum(p[0] for p in parts)), "flops": float(sum(p[1] for p in parts))}


# --------------------------------------------------------------------------
# the same runs in plain torch, 64 bits
# --------------------------------------------------------------------------
def _shape_functions(etype, dev):
    """Weights [q], shape functions [q][n], natural derivatives [q][n][3]."""
    f = dict(dtype=torch.float64, device=dev)
    if etype == TET4:
        d = torch.tensor([[-1, -1, -1], [0, 1, 0], [0, 0, 1], [1, 0, 0]], **f)
        return torch.full((1,), 1 / 6, **f), torch.full((1, 4), 0.25, **f), d[None]
    bits = [((b & 1), (b >> 1) & 1, b >> 2) for b in _CUBE]
    s = torch.tensor(bits, **f) * 2 - 1
    g = torch.tensor([(q & 1, (q >> 1) & 1, q >> 2) for q in range(8)], **f) * 2 - 1
    t = 1 + s[None] * g[:, None] / math.sqrt(3.0)  # [q][n][3]
    N = t.prod(2) / 8
    d = torch.stack([s[None, :, i] * t.prod(2) / t[:, :, i] / 8 for i in range(3)], 2)
    return torch.ones(8, **f), N, d


def _inverse(m):
    """Determinant and inverse of [...][3][3]."""
    a, b, c = m[..., 0, :], m[..., 1, :], m[..., 2, :]
    r = torch.stack([torch.linalg.cross(b, c), torch.linalg.cross(c, a),
                     torch.linalg.cross(a, b)], -1)
    det = (a * r[..., 0]).sum(-1)
    return det, r / det[..., None, None]


def _mul(a, b):
    """[...][i][k] [...][k][j]."""
    return sum(a[..., :, k, None] * b[..., None, k, :] for k in range(a.shape[-1]))


def _dt_critical(p, X, conn, lam, mu, rho):
    x = X[conn]
    if p["etype"] == HEX8:
        ed = [(0, 1), (1, 2), (2, 3), (3, 0), (0, 4), (1, 5), (2, 6), (3, 7), (4, 5), (5, 6),
              (6, 7), (7, 4)]
        h = torch.stack([(x[:, a] - x[:, b]).norm(dim=1) for a, b in ed]).amin(0)
    else:
        def area(a, b, c):
            return torch.linalg.cross(x[:, b] - x[:, a], x[:, c] - x[:, a]).norm(dim=1) / 2
        vol = (torch.linalg.cross(x[:, 1] - x[:, 0], x[:, 2] - x[:, 0])
               * (x[:, 3] - x[:, 0])).sum(1).abs() / 6
        h = 2 * 3 * vol / (area(0, 1, 2) + area(1, 3, 2) + area(0, 2, 3) + area(0, 1, 3))
    return float((h / torch.sqrt((lam + 2 * mu) / rho)).min())


def _simulate(p, steps):
    """`steps` explicit steps: u, v and the internal force."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    f64 = dict(dtype=torch.float64, device=dev)
    X = torch.as_tensor(p["mesh"].nodes, **f64)
    conn = torch.as_tensor(p["mesh"].conn, device=dev).long()
    mat, law = p["mat"], p["law"]
    E = torch.as_tensor(mat.get("E_el", mat["E"]), **f64)
    nu = torch.as_tensor(mat.get("nu_el", mat["nu"]), **f64)
    lam, mu = nu * E / ((1 + nu) * (1 - 2 * nu)), E / (2 * (1 + nu))
    dt = 0.5 * _dt_critical(p, X, conn, lam, mu, mat["rho"])
    w, N, dN = _shape_functions(p["etype"], dev)
    nel, nnpe = conn.shape
    free = 1 - torch.as_tensor(p["blocked"], **f64)
    eye = torch.eye(3, **f64)
    mass = torch.zeros(X.shape[0], **f64)
    B, wJ = [], []  # per Gauss point: dN/dX [e][n][3] and w det J [e]
    for q in range(w.numel()):
        J = sum(dN[q, n][:, None] * X[conn[:, n]][:, None, :] for n in range(nnpe))
        det, Ji = _inverse(J)
        B.append(torch.stack([(Ji * dN[q, n]).sum(-1) for n in range(nnpe)], 1))
        wJ.append(det * w[q])
        for n in range(nnpe):
            mass.index_add_(0, conn[:, n], mat["rho"] * N[q, n] * wJ[q])
    if lam.dim():
        lam, mu = lam[:, None, None], mu[:, None, None]
    eps_p = [torch.zeros(nel, 3, 3, **f64) for _ in wJ] if law == PLASTIC else None
    iso = [torch.zeros(nel, **f64) for _ in wJ] if law == PLASTIC else None

    def stress(q, g):
        """The tensor whose product with dN/dX is the nodal force."""
        if law in (ELASTIC, PLASTIC):
            e = (g + g.transpose(1, 2)) / 2
            if law == PLASTIC:
                e = e - eps_p[q]
            s = lam * e.diagonal(dim1=1, dim2=2).sum(1)[:, None, None] * eye + 2 * mu * e
            if law == ELASTIC:
                return s
            dev_s = s - s.diagonal(dim1=1, dim2=2).sum(1)[:, None, None] / 3 * eye
            eff = torch.sqrt(1.5 * (dev_s * dev_s).sum((1, 2)))
            dp = ((eff - iso[q] - mat["sigma_y"]) / (3 * mu + mat["h"])).clamp_min(0)
            iso[q] += mat["h"] * dp
            de = dev_s * (1.5 * dp / eff.clamp_min(1e-300))[:, None, None]
            eps_p[q] += de
            return s - 2 * mu * de
        F = g + eye
        C = _mul(F.transpose(1, 2), F)
        if law == ELASTIC_FD:
            e = (_mul(g.transpose(1, 2), g) + g + g.transpose(1, 2)) / 2
            S = lam * e.diagonal(dim1=1, dim2=2).sum(1)[:, None, None] * eye + 2 * mu * e
        else:
            J, _ = _inverse(F)
            S = mu * eye + (lam * torch.log(J)[:, None, None] - mu) * _inverse(C)[1]
        return _mul(F, S)

    u, a = torch.zeros_like(X), torch.zeros_like(X)
    v = torch.as_tensor(p["velocity"], **f64).clone()
    for _ in range(steps):
        u += free * (dt * v + 0.5 * dt * dt * a)
        v += free * dt * a
        ue = u[conn]
        f = torch.zeros(nel, nnpe, 3, **f64)
        for q in range(len(wJ)):
            g = sum(ue[:, n, :, None] * B[q][:, n, None, :] for n in range(nnpe))
            P = stress(q, g) * wJ[q][:, None, None]
            f += sum(P[:, None, :, j] * B[q][:, :, j, None] for j in range(3))
        fint = torch.zeros_like(X).index_add_(0, conn.reshape(-1), -f.reshape(-1, 3))
        x = free * (fint / mass[:, None] - a)
        a += x
        v += 0.5 * dt * x
    return [t.cpu() for t in (u, v, fint)]


def exact(case, seed):
    if case["kind"] == "model":
        cells = (case["nx"], case["ny"], case["nz"])
        return _simulate(_inputs(case["etype"], cells, case["law"], seed, case["per_element"]),
                         case["steps"])
    return [_simulate(p, case["steps"] + (3 * k if case["kind"] == "serve" else 0))
            for k, p in enumerate(_instances(case, seed))]
