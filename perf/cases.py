"""Work that users of the shell library have it do, through its Python API.

A case is a dict of plain values.  prepare() makes what a program has in hand
before the call (mesh, equation numbers, FEMM, matrices resident on the
device), run() makes one pass through the public entry points, exact() gives
the same outputs in 64 bits from the element formulas alone (torch), and
work() the bytes and operations of one pass.  Kinds of cases:

  stiffness   stiffness(femm, assembler, ...) with the CSR matrix on the host
  request     one served job from its mesh to its matrices (serve.execute)
  explicit    the central-difference loop on matrices that are on the device
  analysis    new stiffness and mass on the device, then the loop
  stable_dt   new stiffness, mass, and omega_max by power iteration
  batch       many independent plates assembled and stepped together
  statics     consistent pressure load, and the stress resultants of every
              element of a displacement field
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "finetoolsflexstructures.jl_amd"))
from flexshell import batch as FB, explicit as FX, fe, femm as FM, material as MT, serve as FSV  # noqa: E402

GAUSS2 = 0.577350269189626
FP64, MIXED, MIXED_F32 = 0, 1, 2

_DEFAULTS = dict(nen=3, layered=False, nx=32, ny=32, shape="plate", edges="clamped", formulation=0, block="free",
                 precision=FP64, steps=0, damped=False, pulse=False, maxit=0, models=0, nmin=0, nmax=0)


def _case(kind, name=None, **kw):
    c = dict(_DEFAULTS, kind=kind, **kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest model of the repository's configurations, a clamped
        # 32 x 32 plate: stiffness for a static solve on the host
        _case("stiffness", "stiffness_t3_32x32", nx=32, ny=32),
        # the cylindrical panel of the repository's benchmark at full size,
        # free-free stiffness handed to a host solver (680 MB of values)
        _case("stiffness", "stiffness_q4_512x512", nen=4, nx=512, ny=512, shape="cylinder", edges="simple"),
        # one served request, a layered shell of ordinary size with an odd
        # mesh: stiffness and mass for a modal solve, the model used once
        _case("request", "request_q4comp_149x83", nen=4, layered=True, nx=149, ny=83, edges="simple"),
        # a short transient of the smallest plate: a loop of many tiny steps
        _case("explicit", "explicit_t3_32x32", nx=32, ny=32, steps=1000, pulse=True),
        # a damped transient of an ordinary panel
        _case("explicit", "explicit_q4_97x61_damped", nen=4, nx=97, ny=61, shape="cylinder", edges="simple",
              steps=500, damped=True),
        # the benchmark's panel from its geometry's stiffness to the state
        # after the first 200 steps (Gaussian initial velocities)
        _case("analysis", "analysis_q4_512x512", nen=4, nx=512, ny=512, shape="cylinder", edges="simple", steps=200),
        # the largest model, a million triangles under a pressure pulse, with
        # probes, on matrices that are on the device already
        _case("explicit", "explicit_t3_1024x512", nx=1024, ny=512, steps=200, pulse=True),
        # the two mixed precisions of the loop
        _case("explicit", "explicit_t3_512x256_mixed_f32", nx=512, ny=256, steps=200, pulse=True,
              precision=MIXED_F32),
        _case("explicit", "explicit_q4_256x200_mixed", nen=4, nx=256, ny=200, shape="cylinder", edges="simple",
              steps=200, precision=MIXED),
        # the stable time step of a new layered design (100 iterations, as the
        # server takes them), with the second transverse-shear formulation
        _case("stable_dt", "stable_dt_t3comp_300x211", layered=True, nx=300, ny=211, formulation=1, maxit=100),
        # many independent plates of unlike sizes, assembled and stepped in
        # one launch per kernel with the step loop in a graph
        _case("batch", "batch_t3_48_models", models=48, nmin=8, nmax=64, steps=300),
        # load vector and stress resultants of a whole plate around a static
        # solution
        _case("statics", "statics_q4_320x257", nen=4, nx=320, ny=257),
    ]


def draw(rng):
    def size(lo, hi, nen):
        e = math.exp(rng.uniform(math.log(lo), math.log(hi))) / (2 if nen == 3 else 1)
        a = rng.uniform(1.0, 3.0)
        ny = max(3, round(math.sqrt(e / a)))
        return max(3, round(e / ny)), ny

    kind = rng.choice(["stiffness", "request", "explicit", "explicit", "analysis", "stable_dt", "batch", "statics"])
    nen = rng.choice([3, 4])
    layered = rng.random() < (1.0 if kind == "request" else 0.4)
    shape = "plate" if layered or kind == "statics" else rng.choice(["plate", "cylinder"])
    hi = {"stiffness": 250e3, "request": 120e3, "explicit": 800e3, "analysis": 250e3, "stable_dt": 250e3,
          "statics": 150e3, "batch": 1e3}[kind]
    nx, ny = size(900, hi, nen)
    c = _case(kind, nen=nen, layered=layered, nx=nx, ny=ny, shape=shape, edges=rng.choice(["clamped", "simple"]))
    if nen == 3 and kind in ("stiffness", "analysis", "stable_dt"):
        c["formulation"] = rng.choice([0, 0, 1])
    if kind == "stiffness":
        c["block"] = rng.choice(["free", "all"])
    if kind == "explicit":
        c["precision"] = rng.choice([FP64, FP64, FP64, MIXED_F32, MIXED])
        c["steps"] = rng.choice([100, 150, 200, 300])
    if kind == "analysis":
        c["steps"] = rng.choice([50, 100, 200])
    if kind in ("explicit", "analysis"):
        c["damped"] = rng.random() < 0.3
        c["pulse"] = rng.random() < 0.5
    if kind == "stable_dt":
        c["maxit"] = rng.choice([30, 60, 100])
    if kind == "batch":
        c.update(nen=3, layered=False, shape="plate", nx=0, ny=0, models=rng.randint(4, 60), nmin=8,
                 nmax=rng.randint(24, 72), steps=rng.choice([100, 200, 300]))
    return c


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------

def _mesh(nen, nx, ny, Lx, Ly, shape, edges, rng):
    """Structured mesh with +-10 % jittered interior nodes: node coordinates,
    connectivity (element columns along y), fixed-dof flags."""
    X, Y = np.meshgrid(np.linspace(0.0, Lx, nx + 1), np.linspace(0.0, Ly, ny + 1))
    x, y = X.ravel(), Y.ravel()
    left, right = x < 1e-9, x > Lx - 1e-9
    low, high = y < 1e-9, y > Ly - 1e-9
    inner = ~(left | right | low | high)
    x, y = x.copy(), y.copy()
    x[inner] += rng.uniform(-0.1, 0.1, inner.sum()) * (Lx / nx)
    y[inner] += rng.uniform(-0.1, 0.1, inner.sum()) * (Ly / ny)
    if shape == "cylinder":  # x is the arc length on a radius of 1
        xyz = np.stack([np.sin(x), y, np.cos(x)], axis=1)
    else:
        xyz = np.stack([x, y, np.zeros_like(x)], axis=1)
    i, j = np.meshgrid(np.arange(nx), np.arange(ny), indexing="ij")
    f = (j * (nx + 1) + i).ravel().astype(np.int64)
    if nen == 4:
        conn = np.stack([f, f + 1, f + nx + 2, f + nx + 1], axis=1)
    else:
        conn = np.empty((2 * f.size, 3), dtype=np.int64)
        conn[0::2] = np.stack([f, f + 1, f + nx + 1], axis=1)
        conn[1::2] = np.stack([f + 1, f + nx + 2, f + nx + 1], axis=1)
    fixed = np.zeros((xyz.shape[0], 6), dtype=bool)
    if edges == "clamped":
        fixed[~inner] = True
    else:
        fixed[left | right, :3] = True
    return xyz, conn, fixed


def _numbers(fixed):
    """Equation numbers: free dofs in node order, then the fixed ones."""
    free = ~fixed
    nf = int(free.sum())
    dn = np.empty(fixed.shape, dtype=np.int64)
    dn[free] = np.arange(nf)
    dn[fixed] = nf + np.arange(fixed.size - nf)
    return dn, nf


def _model(case, seed):
    """One model: mesh, numbering, homogeneous or layered section."""
    rng = np.random.default_rng([seed, 11])
    nen = case["nen"]
    if case["layered"]:
        Ly = 0.5
        Lx = Ly * case["nx"] / case["ny"]
    elif case["shape"] == "cylinder":
        Lx, Ly = math.pi / 3, 2.0
    else:
        Ly = 1.0
        Lx = Ly * case["nx"] / case["ny"]
    xyz, conn, fixed = _mesh(nen, case["nx"], case["ny"], Lx, Ly, case["shape"], case["edges"], rng)
    dn, nf = _numbers(fixed)
    m = dict(nen=nen, xyz=xyz, conn=conn, fixed=fixed, dofnums=dn, nf=nf, layered=case["layered"],
             formulation=case["formulation"], stab_c=5 / 12 / 1.5 if nen == 3 else 0.1, h=min(Lx / case["nx"], Ly / case["ny"]))
    if case["layered"]:
        n = int(rng.integers(3, 9))
        m["plies"] = [(0.125e-3, float(a)) for a in rng.choice([0.0, 45.0, -45.0, 90.0], n)]
        m["lamina"] = dict(E1=140e9 * rng.uniform(0.9, 1.1), E2=10e9, G12=5e9, nu12=0.3, rho=1600.0)
    else:
        m.update(E=70e9 * rng.uniform(0.9, 1.1), nu=0.33, rho=2700.0, t=0.005 * rng.uniform(0.9, 1.1))
    return m


def _loads(case, m, seed):
    """Initial velocities of the free translations, load vector, load history,
    probed dofs."""
    rng = np.random.default_rng([seed, 12])
    V0 = np.zeros(m["nf"])
    trans = m["dofnums"][:, :3][~m["fixed"][:, :3]]
    V0[trans] = rng.normal(0.0, 1e-3, trans.size)
    F = np.zeros(m["nf"])
    g = np.zeros(case["steps"] + 1)
    probes = np.zeros(0, dtype=np.int64)
    if case["pulse"]:
        c = m["xyz"][rng.integers(0, m["xyz"].shape[0])]
        p = 1e4 * np.exp(-((m["xyz"] - c) ** 2).sum(axis=1) / (2 * 0.1 ** 2)) * m["h"] ** 2
        up = ~m["fixed"][:, 2]
        F[m["dofnums"][up, 2]] = p[up]
        g[: max(2, case["steps"] // 5)] = 1.0
        probes = np.sort(rng.choice(m["nf"], size=min(64, m["nf"]), replace=False)).astype(np.int64)
    return V0, F, g, probes


def _dt(m, seed):
    """A time step below the stability limit, from the largest eigenvalue of
    sampled element pencils (an upper bound of the model's, with a margin for
    the elements that are not in the sample)."""
    pick = np.random.default_rng([seed, 13]).choice(m["conn"].shape[0], size=min(128, m["conn"].shape[0]), replace=False)
    sub = dict(m, conn=m["conn"][pick])
    nrm = _normals(m) if m["xyz"].shape[0] < 20000 else None
    if nrm is None:  # normals of the sampled elements' nodes: smooth surfaces
        nrm = np.zeros_like(m["xyz"])
        nrm[:, 2] = 1.0
        if abs(m["xyz"][:, 2]).max() > 0:
            nrm[:, 0], nrm[:, 2] = m["xyz"][:, 0], m["xyz"][:, 2]
    Ke = _element_matrices(sub, nrm, "cpu")
    tm, rm = _element_masses(sub)
    d = np.tile(np.repeat(np.stack([tm, rm], axis=1), 3, axis=1), (1, m["nen"])) ** -0.5
    w2 = np.linalg.eigvalsh(Ke.numpy() * d[:, :, None] * d[:, None, :]).max()
    return 0.75 * 2 / math.sqrt(w2)


def _layup(m):
    L = m["lamina"]
    mat = MT.lamina_material(L["rho"], L["E1"], L["E2"], L["nu12"], L["G12"], L["G12"], L["E2"] / 2.6)
    return MT.CompositeLayup("layup", [MT.Ply(f"ply{k}", mat, t, a) for k, (t, a) in enumerate(m["plies"])], np.eye(3))


def _femm(m):
    if m["layered"]:
        f = FM.make(m["conn"], _layup(m))
    else:
        f = FM.make(m["conn"], MT.MatDeforElastIso(m["E"], m["nu"], m["rho"]), thickness=m["t"])
    f.transv_shear_formulation = m["formulation"]
    return f


def _field(m):
    d = fe.DofField(m["xyz"].shape[0])
    d.is_fixed[:] = m["fixed"]
    return d.numberdofs()


def _batch_models(case, seed):
    rng = np.random.default_rng([seed, 14])
    sizes = np.random.default_rng([case["models"], case["nmin"], case["nmax"]])  # the case's, for every seed
    out = []
    for k in range(case["models"]):
        n = int(sizes.integers(case["nmin"], case["nmax"] + 1))
        Lx = float(rng.uniform(1.0, 4.0))
        xyz, conn, fixed = _mesh(3, n, n, Lx, 1.0, "plate", "clamped" if sizes.random() < 0.5 else "simple", rng)
        dn, nf = _numbers(fixed)
        out.append(dict(nen=3, xyz=xyz, conn=conn, fixed=fixed, dofnums=dn, nf=nf, layered=False, formulation=0,
                        stab_c=5 / 12 / 1.5, E=float(np.exp(rng.uniform(np.log(1e9), np.log(3e11)))),
                        nu=float(rng.uniform(0.2, 0.4)), rho=float(rng.uniform(1000.0, 8000.0)),
                        t=float(np.exp(rng.uniform(np.log(0.002), np.log(0.05)))), h=min(Lx, 1.0) / n))
    return out


def _batch_inputs(case, seed):
    ms = _batch_models(case, seed)
    dts = np.array([_dt(m, seed) for m in ms])
    V0 = np.concatenate([_loads(case, m, seed + k)[0] for k, m in enumerate(ms)])
    return ms, dts, V0


# ---------------------------------------------------------------------------
# the passes
# ---------------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        ms, dts, V0 = _batch_inputs(case, seed)
        b = FB.ShellBatch([dict(xyz=m["xyz"], conn=m["conn"], dchi=_field(m), t=m["t"],
                                material=MT.MatDeforElastIso(m["E"], m["nu"], m["rho"])) for m in ms])
        b.assemble_device()
        b.mass()
        n = len(ms)
        return dict(case=case, batch=b, dts=dts, cd=np.zeros(n), U0=np.zeros(b.nfree), V0=V0, F=np.zeros(b.nfree),
                    g=np.zeros((case["steps"] + 1, n)))
    m = _model(case, seed)
    d = _field(m)
    s = dict(case=case, m=m, d=d)
    if kind == "request":
        s["ctx"] = FSV.request_context()
        s["req"] = FSV.Request(0, FSV.MODAL, dict(xyz=m["xyz"], conn=m["conn"], dchi=d, layup=_layup(m)))
        return s
    f = s["femm"] = _femm(m)
    f.associategeometry(m["xyz"])
    if kind == "statics":
        rng = np.random.default_rng([seed, 15])
        s["u"] = rng.normal(0.0, 1e-4, (m["xyz"].shape[0], 6))
        return s
    if kind == "stiffness":
        s["asm"] = FM.SysmatAssemblerFFBlock(m["nf"]) if case["block"] == "free" else FM.SysmatAssemblerSparseCSRSymm()
        return s
    s["asm"] = FM.SysmatAssemblerHIP()
    f.stiffness(s["asm"], m["xyz"], None, None, d)
    f.mass(s["asm"], m["xyz"], d)
    if kind == "stable_dt":
        s["v0"] = np.random.default_rng([seed, 16]).standard_normal(m["nf"])
        return s
    s["V0"], s["F"], s["g"], s["probes"] = _loads(case, m, seed)
    s["U0"] = np.zeros(m["nf"])
    s["dt"] = _dt(m, seed)
    s["cdamp"] = 0.02 * 2 * (0.05 / s["dt"]) if case["damped"] else 0.0
    return s


def _csr_out(K):
    return {"rowptr": K.indptr, "colval": K.indices, "nzval": K.data}


def _step(s):
    c = s["case"]
    r = FX.run(s["femm"]._model, s["cdamp"], s["U0"], s["V0"], s["dt"], c["steps"], s["F"], s["g"], s["probes"], 10,
               c["precision"])
    return {"U": r["U"], "V": r["V"], "probes": r["probes"]}


def run(s):
    c, kind = s["case"], s["case"]["kind"]
    if kind == "batch":
        r = s["batch"].explicit(s["dts"], s["cd"], s["U0"], s["V0"], s["F"], s["g"], c["steps"])
        return {"U": r["U"], "V": r["V"]}
    m, d = s["m"], s["d"]
    if kind == "stiffness":
        return _csr_out(s["femm"].stiffness(s["asm"], m["xyz"], None, None, d))
    if kind == "request":
        r = FSV.execute(s["req"], s["ctx"])
        return dict(_csr_out(r["K"]), M=r["M"])
    if kind == "explicit":
        return _step(s)
    if kind == "analysis":
        s["femm"].stiffness(s["asm"], m["xyz"], None, None, d)
        s["femm"].mass(s["asm"], m["xyz"], d)
        return _step(s)
    if kind == "stable_dt":
        f = s["femm"]
        f.stiffness(s["asm"], m["xyz"], None, None, d)
        M = f.mass(FM.SysmatAssemblerFFBlock(FM.SysmatAssemblerSparseDiag(), m["nf"], m["nf"]), m["xyz"], d)
        return {"omega": FX.omega_max(f, s["v0"], c["maxit"]), "M": M.diagonal()}
    if kind == "statics":
        F = s["femm"].distribloads(m["xyz"], d, [0.0, 0.0, 1e3, 0.0, 0.0, 0.0])
        out, loc = s["femm"].resultants(m["xyz"], s["u"], outputcsys=np.eye(3))
        return {"F": F, "out": out, "loc": loc}
    raise ValueError(kind)


# ---------------------------------------------------------------------------
# bytes and operations
# ---------------------------------------------------------------------------

def _stored(nen, nx, ny):
    """(elements, nodes, entries of the all-dof matrix) of a structured mesh."""
    N = (nx + 1) * (ny + 1)
    pairs = nx * (ny + 1) + ny * (nx + 1) + nx * ny * (1 if nen == 3 else 2)
    return nx * ny * (2 if nen == 3 else 1), N, 36 * (N + 2 * pairs)


def work(case):
    kind, nen = case["kind"], case["nen"]
    if kind == "batch":
        n = (case["nmin"] + case["nmax"]) // 2
        E, N, nnz = (v * case["models"] for v in _stored(3, n, n))
    else:
        E, N, nnz = _stored(nen, case["nx"], case["ny"])
    npt = 1 if nen == 3 else 4
    k = 6 * nen
    # mesh, normals in; values out; rows of B D B per point, upper half
    asm = dict(bytes=4 * nen * E + 49 * N + 8 * nnz, flops=E * npt * (8 * k * (k + 1) + 8 * 8 * k))
    # the symmetric matrix's upper half, U and V in and out, the mass
    step = dict(bytes=4 * nnz + 40 * 6 * N, flops=2 * nnz + 60 * N)
    if kind in ("stiffness", "request"):
        return dict(bytes=asm["bytes"] + 12 * nnz, flops=asm["flops"])
    if kind in ("explicit", "batch"):
        return {q: case["steps"] * step[q] for q in step}
    if kind == "analysis":
        return {q: asm[q] + case["steps"] * step[q] for q in step}
    if kind == "stable_dt":
        return {q: asm[q] + (case["maxit"] + 1) * step[q] for q in step}
    if kind == "statics":
        return dict(bytes=4 * nen * E + 145 * N + 88 * npt * E, flops=1500 * npt * E)
    raise ValueError(kind)


# ---------------------------------------------------------------------------
# the same outputs in 64 bits
# ---------------------------------------------------------------------------

def _frames(J):
    """Element frames (columns e1, e2, e3) of tangent matrices ... x 3 x 2."""
    e1 = J[..., 0] / J[..., 0].norm(dim=-1, keepdim=True)
    n = torch.linalg.cross(e1, J[..., 1])
    e3 = n / n.norm(dim=-1, keepdim=True)
    return torch.stack([e1, torch.linalg.cross(e3, e1), e3], dim=-1)


def _shape(xi, eta):
    N = torch.tensor([(1 - xi) * (1 - eta), (1 + xi) * (1 - eta), (1 + xi) * (1 + eta), (1 - xi) * (1 + eta)],
                     dtype=torch.float64) / 4
    g = torch.tensor([[-(1 - eta), -(1 - xi)], [1 - eta, -(1 + xi)], [1 + eta, 1 + xi], [-(1 + eta), 1 - xi]],
                     dtype=torch.float64) / 4
    return N, g


def _normals(m):
    X = torch.from_numpy(m["xyz"][m["conn"]])
    nrm = torch.zeros(m["xyz"].shape[0], 3, dtype=torch.float64)
    conn = torch.from_numpy(m["conn"])
    if m["layered"]:
        nrm[:, 2] = 1.0  # the layup's constant coordinate system
    elif m["nen"] == 3:
        e3 = _frames(torch.stack([X[:, 1] - X[:, 0], X[:, 2] - X[:, 0]], dim=-1))[..., 2]
        for a in range(3):
            nrm.index_add_(0, conn[:, a], e3)
    else:
        for a, (xi, eta) in enumerate([(-1, -1), (1, -1), (1, 1), (-1, 1)]):
            J = torch.einsum("eak,ap->ekp", X, _shape(xi, eta)[1])
            nrm.index_add_(0, conn[:, a], torch.linalg.cross(J[..., 0], J[..., 1]))
    return (nrm / nrm.norm(dim=1, keepdim=True)).numpy()


def _plane_stress(D):
    return D[:2, :2] - np.outer(D[:2, 2], D[2, :2]) / D[2, 2]


def _section(m):
    """8 x 8 constitutive matrix (membrane, bending, shear without its
    stabilisation factor) per element frame of a homogeneous section, or A, B,
    D, H of a laminate in its own frame; thickness; masses per area."""
    if not m["layered"]:
        E, nu, t = m["E"], m["nu"], m["t"]
        Q = E / (1 - nu * nu) * np.array([[1, nu, 0], [nu, 1, 0], [0, 0, (1 - nu) / 2]])
        H = 5 / 6 * E / 2 / (1 + nu) * np.eye(2)
        return t * Q, 0 * Q, t ** 3 / 12 * Q, t * H, t, m["rho"] * t, m["rho"] * t ** 3 / 12
    L = m["lamina"]
    C = np.zeros((6, 6))
    C[:3, :3] = [[1 / L["E1"], -L["nu12"] / L["E1"], -L["nu12"] / L["E1"]], [-L["nu12"] / L["E1"], 1 / L["E2"], 0],
                 [-L["nu12"] / L["E1"], 0, 1 / L["E2"]]]
    D6 = np.linalg.inv(C[:3, :3])
    Q = np.zeros((3, 3))
    Q[:2, :2] = _plane_stress(D6)
    Q[2, 2] = L["G12"]
    S = np.diag([L["G12"], L["E2"] / 2.6])
    A, B, D, H = np.zeros((3, 3)), np.zeros((3, 3)), np.zeros((3, 3)), np.zeros((2, 2))
    tl = sum(t for t, _ in m["plies"])
    z, md, mi = -tl / 2, 0.0, 0.0
    for t, a in m["plies"]:
        ze = z + t
        c, s = math.cos(math.radians(a)), math.sin(math.radians(a))
        T = np.array([[c * c, s * s, -2 * c * s], [s * s, c * c, 2 * c * s], [c * s, -c * s, c * c - s * s]])
        R = np.array([[c, -s], [s, c]])
        A += (ze - z) * T @ Q @ T.T
        B += (ze ** 2 - z ** 2) / 2 * T @ Q @ T.T
        D += (ze ** 3 - z ** 3) / 3 * T @ Q @ T.T
        H += 5 / 4 * (ze - z - 4 / 3 * (ze ** 3 - z ** 3) / tl ** 2) * R.T @ S @ R
        md += (ze - z) * L["rho"]
        mi += (ze ** 3 - z ** 3) * L["rho"] / 3
        z = ze
    return A, B, D, H, tl, md, mi


def _constitutive(m, EG):
    """E x 8 x 8 constitutive matrices in the element frames, thickness."""
    A, B, D, H, t, _, _ = (torch.as_tensor(v, dtype=torch.float64, device=EG.device) for v in _section(m))
    out = torch.zeros(EG.shape[0], 8, 8, dtype=torch.float64, device=EG.device)
    if m["layered"]:  # layup frame = global axes: angle of the frame's projection
        c0 = EG[:, 0, :2] / EG[:, 0, :2].norm(dim=1, keepdim=True)
        c1 = EG[:, 1, :2] / EG[:, 1, :2].norm(dim=1, keepdim=True)
        c = (c0[:, 0] + c1[:, 1]) / 2
        s = (c1[:, 0] - c0[:, 1]) / 2
        Ti = torch.stack([c * c, s * s, 2 * c * s, s * s, c * c, -2 * c * s, -c * s, c * s, c * c - s * s],
                         dim=1).reshape(-1, 3, 3)
        Tt = torch.stack([c, -s, s, c], dim=1).reshape(-1, 2, 2)
        rot = lambda M, T: torch.matmul(torch.matmul(T, M), T.transpose(1, 2).contiguous())  # noqa: E731
        out[:, :3, :3], out[:, 3:6, 3:6] = rot(A, Ti), rot(D, Ti)
        out[:, :3, 3:6] = rot(B, Ti)
        out[:, 3:6, :3] = out[:, :3, 3:6].transpose(1, 2)
        out[:, 6:, 6:] = rot(H, Tt.transpose(1, 2).contiguous())
    else:
        out[:, :3, :3], out[:, 3:6, 3:6], out[:, 6:, 6:] = A, D, H
    return out, t


def _transforms(EG, nrm, gN):
    """Tae (nodal to element) and Tga (global to nodal) of E elements."""
    E, nn = nrm.shape[0], nrm.shape[1]
    nk = torch.einsum("eki,eak->eai", EG, nrm)
    r = torch.stack([-nk[..., 1], nk[..., 0], torch.zeros_like(nk[..., 0])], dim=-1)
    na = r.norm(dim=-1)
    u = r / na.clamp(min=1e-300)[..., None]
    Z = torch.zeros_like(na)
    S = torch.stack([Z, -r[..., 2], r[..., 1], r[..., 2], Z, -r[..., 0], -r[..., 1], r[..., 0], Z],
                    dim=-1).reshape(E, nn, 3, 3)
    I = torch.eye(3, dtype=torch.float64, device=EG.device)
    uu = u[..., :, None] * u[..., None, :]
    A = torch.cos(na)[..., None, None] * (I - uu) + (torch.sin(na) / na.clamp(min=1e-300))[..., None, None] * S + uu
    A = torch.where((na > 1e-12)[..., None, None], A, I)
    kd = 6 * nn
    Tae = torch.zeros(E, kd, kd, dtype=torch.float64, device=EG.device)
    Tga = torch.zeros_like(Tae)
    for i in range(nn):
        o = 6 * i
        Q = torch.einsum("ekr,eck->erc", A[:, i], EG)
        Tga[:, o:o + 3, o:o + 3] = Q
        Tga[:, o + 3:o + 6, o + 3:o + 6] = Q
        Ai, a33 = A[:, i], A[:, i, 2, 2]
        Tae[:, o:o + 3, o:o + 3] = Ai
        Tae[:, o + 3:o + 5, o + 3:o + 5] = Ai[:, :2, :2] - Ai[:, :2, 2, None] * Ai[:, None, :2, 2] / a33[:, None, None]
        for j in range(nn):
            a3 = (Ai[:, 1] * gN[:, j, 0, None] - Ai[:, 0] * gN[:, j, 1, None]) / 2
            for q in (0, 1):
                Tae[:, o + 3 + q, 6 * j:6 * j + 3] += (Ai[:, q, 2] / a33)[:, None] * a3
    return Tae, Tga


def _strain_rows(gN):
    """Membrane and bending rows of B."""
    E, nn = gN.shape[0], gN.shape[1]
    B = torch.zeros(E, 6, 6 * nn, dtype=torch.float64, device=gN.device)
    for i in range(nn):
        o, gx, gy = 6 * i, gN[:, i, 0], gN[:, i, 1]
        B[:, 0, o], B[:, 1, o + 1], B[:, 2, o], B[:, 2, o + 1] = gx, gy, gy, gx
        B[:, 3, o + 4], B[:, 4, o + 3], B[:, 5, o + 3], B[:, 5, o + 4] = gx, -gy, -gx, gy
    return B


def _t3_shear(ec, area, s, p, q):
    B = torch.zeros(ec.shape[0], 2, 18, dtype=torch.float64, device=ec.device)
    a, b = (ec[:, p] - ec[:, s]).unbind(1)
    c, d = (ec[:, q] - ec[:, s]).unbind(1)
    k = 1 / (2 * area)
    for node, row0, row1 in ((s, (b - d, 0 * a, area), (c - a, -area, 0 * a)),
                             (p, (d, -b * d / 2, a * d / 2), (-c, b * c / 2, -a * c / 2)),
                             (q, (-b, b * d / 2, -b * c / 2), (a, -a * d / 2, a * c / 2))):
        for w in range(3):
            B[:, 0, 6 * node + 2 + w] += k * row0[w]
            B[:, 1, 6 * node + 2 + w] += k * row1[w]
    return B


def _q4_shear(ec, r, s):
    """Assumed transverse-shear strains of the four-node element, from the
    covariant strains at the mid-sides of its edges.  The element takes the
    interpolation and its scales at the mirrored point (-r, -s)."""
    B = torch.zeros(ec.shape[0], 2, 24, dtype=torch.float64, device=ec.device)
    x, y = ec[..., 0], ec[..., 1]
    g = _shape(r, s)[1].to(ec.device)
    J = torch.einsum("eak,ap->ekp", ec, g)
    A, Bn = J[:, :, 0].norm(dim=1), J[:, :, 1].norm(dim=1)
    Jm = torch.einsum("eak,ap->ekp", ec, _shape(-r, -s)[1].to(ec.device))
    ca, sa, cb, sb = J[:, 0, 0] / A, J[:, 1, 0] / A, J[:, 0, 1] / Bn, J[:, 1, 1] / Bn
    det = J[:, 0, 0] * J[:, 1, 1] - J[:, 0, 1] * J[:, 1, 0]
    P, Q = 4 * Jm[:, :, 0].norm(dim=1), 4 * Jm[:, :, 1].norm(dim=1)
    # strain along r from the edges 1-2 and 4-3, along s from the edges 1-4 and
    # 2-3, interpolated linearly
    lines = ((0, 1, 1 + s, 0), (3, 2, 1 - s, 0), (0, 3, 1 + r, 1), (1, 2, 1 - r, 1))
    for i, j, w, along in lines:
        dx, dy = x[:, j] - x[:, i], y[:, j] - y[:, i]
        scale = (Q if along == 0 else P) / (16 * det)
        for row, f in ((0, sb if along == 0 else -sa), (1, -cb if along == 0 else ca)):
            k = f * scale * w
            B[:, row, 6 * j + 2] += k
            B[:, row, 6 * i + 2] -= k
            for n in (i, j):
                B[:, row, 6 * n + 3] -= k * dy / 2
                B[:, row, 6 * n + 4] += k * dx / 2
    return B


def _points(m, nrm, conn, dev):
    """Integration points of the elements: (weight, B T of the 8 strain rows
    per shear set, T, constitutive matrix, frame, stabilisation, gN)."""
    X = torch.as_tensor(m["xyz"], device=dev)[conn]
    nv = torch.as_tensor(nrm, device=dev)[conn]
    if m["nen"] == 3:
        J = torch.stack([X[:, 1] - X[:, 0], X[:, 2] - X[:, 0]], dim=-1)
        EG = _frames(J)
        ec = torch.einsum("eak,ekp->eap", X - X[:, :1], EG[..., :2])
        a, b = ec[:, 1].unbind(1)
        c, d = ec[:, 2].unbind(1)
        area = (a * d - b * c) / 2
        gN = torch.stack([b - d, c - a, d, -c, -b, a], dim=1).reshape(-1, 3, 2) / (2 * area)[:, None, None]
        sh = [_t3_shear(ec, area, *o) for o in ((0, 1, 2), (1, 2, 0), (2, 0, 1))]
        if m["formulation"] == 0:
            sh = [(sh[0] + sh[1] + sh[2]) / 3]
        D, t = _constitutive(m, EG)
        stab = t * t / (t * t + m["stab_c"] * 2 * area)
        yield area, _strain_rows(gN), sh, _transforms(EG, nv, gN), D, EG, stab
        return
    h2 = ((X[:, 1:] - X[:, :1]) ** 2).sum(dim=2).max(dim=1).values
    for xi in (-GAUSS2, GAUSS2):
        for eta in (-GAUSS2, GAUSS2):
            g = _shape(xi, eta)[1].to(dev)
            J = torch.einsum("eak,ap->ekp", X, g)
            w = torch.linalg.cross(J[..., 0], J[..., 1]).norm(dim=1)
            EG = _frames(J)
            ec = torch.einsum("eak,ekp->eap", X - X.mean(dim=1, keepdim=True), EG[..., :2])
            J2 = torch.einsum("ekp,ekq->epq", EG[..., :2], J)
            det = J2[:, 0, 0] * J2[:, 1, 1] - J2[:, 0, 1] * J2[:, 1, 0]
            inv = torch.stack([J2[:, 1, 1], -J2[:, 0, 1], -J2[:, 1, 0], J2[:, 0, 0]], dim=1).reshape(-1, 2, 2)
            gN = torch.einsum("ap,epq->eaq", g, inv / det[:, None, None])
            D, t = _constitutive(m, EG)
            stab = t * t / (t * t + m["stab_c"] * h2)
            yield w, _strain_rows(gN), [_q4_shear(ec, xi, eta)], _transforms(EG, nv, gN), D, EG, stab


def _element_matrices(m, nrm, dev, chunk=32768):
    """Element stiffness matrices, E x k x k."""
    nen, kd = m["nen"], 6 * m["nen"]
    conn_all = torch.as_tensor(m["conn"], device=dev)
    out = torch.empty(conn_all.shape[0], kd, kd, dtype=torch.float64, device=dev)
    for lo in range(0, conn_all.shape[0], chunk):
        conn = conn_all[lo:lo + chunk]
        nv = torch.as_tensor(nrm, device=dev)[conn]
        K = torch.zeros(conn.shape[0], kd, kd, dtype=torch.float64, device=dev)
        for w, B6, shears, (Tae, Tga), D, EG, stab in _points(m, nrm, conn, dev):
            T = Tae if nen == 3 else torch.matmul(Tae, Tga)
            for k, Bs in enumerate(shears):
                BT = torch.matmul(torch.cat([B6 if k == 0 else 0 * B6, Bs], dim=1), T)
                Dw = D.clone()
                Dw[:, 6:, 6:] *= (stab / len(shears))[:, None, None]
                K += w[:, None, None] * torch.matmul(BT.transpose(1, 2).contiguous(), torch.matmul(Dw, BT))
        rot = [6 * a + 3 + q for q in range(2) for a in range(nen)]
        if nen == 3:  # drilling in the nodal basis
            kavg = K[:, rot, rot].mean(dim=1)
            for a in range(3):
                K[:, 6 * a + 5, 6 * a + 5] += kavg
            K = torch.matmul(Tga.transpose(1, 2).contiguous(), torch.matmul(K, Tga))
        else:
            s = 0.0
            for a in range(4):
                R = K[:, 6 * a + 3:6 * a + 6, 6 * a + 3:6 * a + 6]
                n = nv[:, a]
                s = s + ((R.diagonal(dim1=1, dim2=2).sum(1) - torch.einsum("ei,eij,ej->e", n, R, n)) / 2).clamp(min=0)
            for a in range(4):
                K[:, 6 * a + 3:6 * a + 6, 6 * a + 3:6 * a + 6] += (s / 4)[:, None, None] * nv[:, a, :, None] * nv[:, a, None, :]
        out[lo:lo + chunk] = K
    return out


def _element_masses(m):
    X = torch.from_numpy(m["xyz"][m["conn"]])
    if m["nen"] == 3:
        area = torch.linalg.cross(X[:, 1] - X[:, 0], X[:, 2] - X[:, 0]).norm(dim=1) / 2
    else:
        area = 0.0
        for xi in (-GAUSS2, GAUSS2):
            for eta in (-GAUSS2, GAUSS2):
                J = torch.einsum("eak,ap->ekp", X, _shape(xi, eta)[1])
                area = area + torch.linalg.cross(J[..., 0], J[..., 1]).norm(dim=1)
    _, _, _, _, _, md, mi = _section(m)
    a = (area / m["nen"]).numpy()
    return md * a, mi * a


def _mass_diag(m):
    tm, rm = _element_masses(m)
    M = np.zeros((m["xyz"].shape[0], 6))
    for a in range(m["nen"]):
        for k, v in ((0, tm), (3, rm)):
            s = np.bincount(m["conn"][:, a], weights=v, minlength=M.shape[0])
            M[:, k:k + 3] += s[:, None]
    d = np.empty(M.size)
    d[m["dofnums"]] = M
    return d


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


class _Operator:
    """K u over the free dofs, element by element."""

    def __init__(self, m, dev):
        self.Ke = _element_matrices(m, _normals(m), dev)
        self.idx = torch.as_tensor(m["dofnums"][m["conn"]].reshape(m["conn"].shape[0], -1), device=dev)
        self.nf, self.nall = m["nf"], m["dofnums"].size

    def __call__(self, u):
        up = torch.cat([u, u.new_zeros(self.nall - self.nf)])
        f = (self.Ke * up[self.idx][:, None, :]).sum(dim=2)
        return torch.zeros_like(up).index_add_(0, self.idx.reshape(-1), f.reshape(-1))[:self.nf]


def _csr_exact(m, block, dev):
    """CSR values (rows and columns ascending) of the assembled matrix."""
    Ke = _element_matrices(m, _normals(m), dev)
    conn = torch.as_tensor(m["conn"], device=dev)
    N, nen = m["xyz"].shape[0], m["nen"]
    I = conn[:, :, None].expand(-1, nen, nen)
    key, inv = torch.unique((I * N + I.transpose(1, 2)).reshape(-1), return_inverse=True)
    blocks = Ke.reshape(-1, nen, 6, nen, 6).permute(0, 1, 3, 2, 4).reshape(-1, 36)
    S = torch.zeros(key.numel(), 36, dtype=torch.float64, device=dev).index_add_(0, inv, blocks)
    del Ke, blocks
    dn = torch.as_tensor(m["dofnums"], device=dev)
    n = m["nf"] if block == "free" else dn.numel()
    r = dn[key // N][:, :, None].expand(-1, 6, 6).reshape(-1)
    c = dn[key % N][:, None, :].expand(-1, 6, 6).reshape(-1)
    keep = (r < n) & (c < n)
    order = torch.argsort(r[keep] * n + c[keep])
    return S.reshape(-1)[keep][order].cpu()


def _march(K, M, dt, cdamp, V0, F, g, steps, probes, stride, dev):
    t = lambda v: torch.as_tensor(v, dtype=torch.float64, device=dev)  # noqa: E731
    M, V, F, dt = t(M), t(V0).clone(), t(F), t(dt)
    U = torch.zeros_like(V)
    C = cdamp * M
    inv = 1 / (M + dt / 2 * C)
    A = inv * (float(g[0]) * F)
    pr = torch.as_tensor(probes, device=dev)
    hist = [U[pr]]
    for n in range(1, steps + 1):
        U = U + (dt * V + dt * dt / 2 * A)
        f = float(g[n]) * F - K(U) - C * (V + dt / 2 * A)
        V = V + dt / 2 * A
        A = inv * f
        V = V + dt / 2 * A
        if n % stride == 0:
            hist.append(U[pr])
    return U.cpu(), V.cpu(), torch.stack(hist).cpu()


def _resultants_exact(m, u, dev):
    conn = torch.as_tensor(m["conn"], device=dev)
    ue = torch.as_tensor(u, device=dev)[conn].reshape(conn.shape[0], -1, 1)
    X = torch.as_tensor(m["xyz"], device=dev)[conn]
    outs = []
    for w, B6, shears, (Tae, Tga), D, EG, stab in _points(dict(m, formulation=0), _normals(m), conn, dev):
        T = torch.matmul(Tae, Tga)
        v = torch.matmul(T, ue)
        if m["layered"] and m["nen"] == 4:
            v = torch.matmul(T, v)  # the layered four-node form takes its displacements through T twice
        e = torch.matmul(torch.cat([B6, shears[0]], dim=1), v)
        D = D.clone()
        D[:, 6:, 6:] *= stab[:, None, None]
        s = torch.matmul(D, e)[..., 0]
        c0 = EG[:, 0, :2] / EG[:, 0, :2].norm(dim=1, keepdim=True)
        c1 = EG[:, 1, :2] / EG[:, 1, :2].norm(dim=1, keepdim=True)
        c, q = (c0[:, 0] + c1[:, 1]) / 2, (c1[:, 0] - c0[:, 1]) / 2
        R = torch.stack([c, q, -q, c], dim=1).reshape(-1, 2, 2)
        parts = []
        for k in (0, 3):
            S = torch.stack([s[:, k], s[:, k + 2], s[:, k + 2], s[:, k + 1]], dim=1).reshape(-1, 2, 2)
            Y = torch.matmul(torch.matmul(R.transpose(1, 2).contiguous(), S), R)
            parts += [Y[:, 0, 0], Y[:, 1, 1], Y[:, 0, 1]]
        sq = torch.matmul(R.transpose(1, 2).contiguous(), s[:, 6:, None])[..., 0]
        outs.append(torch.stack(parts + [sq[:, 0], sq[:, 1]], dim=1))
    if m["nen"] == 3:
        loc = X.mean(dim=1)[:, None]
    else:
        loc = torch.stack([torch.einsum("eak,a->ek", X, _shape(xi, eta)[0].to(dev)) for xi in (-GAUSS2, GAUSS2)
                           for eta in (-GAUSS2, GAUSS2)], dim=1)
    return torch.stack(outs, dim=1).cpu(), loc.cpu()


def _pressure_exact(m):
    """Consistent nodal loads of 1e3 Pa along z (triangles: a constant
    intensity; quadrilaterals: the two by two rule)."""
    X = torch.from_numpy(m["xyz"][m["conn"]])
    F = torch.zeros(m["xyz"].shape[0], dtype=torch.float64)
    if m["nen"] == 3:
        shares = [torch.linalg.cross(X[:, 1] - X[:, 0], X[:, 2] - X[:, 0]).norm(dim=1) / 6] * 3
    else:
        shares = [0.0] * 4
        for xi in (-GAUSS2, GAUSS2):
            for eta in (-GAUSS2, GAUSS2):
                N, g = _shape(xi, eta)
                J = torch.einsum("eak,ap->ekp", X, g)
                w = torch.linalg.cross(J[..., 0], J[..., 1]).norm(dim=1)
                shares = [s + N[a] * w for a, s in enumerate(shares)]
    for a, s in enumerate(shares):
        F.index_add_(0, torch.from_numpy(m["conn"][:, a].copy()), s)
    p = np.zeros((m["xyz"].shape[0], 6))
    p[:, 2] = 1e3 * F.numpy()
    out = np.empty(p.size)
    out[m["dofnums"]] = p
    return out[:m["nf"]]


def exact(case, seed):
    kind, dev = case["kind"], _device()
    _, _, nnz = _stored(case["nen"], max(case["nx"], 1), max(case["ny"], 1))
    if dev == "cpu" and nnz * max(1, case["steps"], case["maxit"]) > 4e9:
        return None
    if kind == "batch":
        ms, dts, V0 = _batch_inputs(case, seed)
        ops, idx, off = [], [], 0
        free = fixed = sum(m["nf"] for m in ms)
        for m in ms:
            op = _Operator(m, dev)
            ops.append(op.Ke)
            idx.append(torch.where(op.idx < m["nf"], op.idx + off, op.idx - m["nf"] + fixed))
            off += m["nf"]
            fixed += op.nall - op.nf
        K = _Operator.__new__(_Operator)
        K.Ke, K.idx, K.nf, K.nall = torch.cat(ops), torch.cat(idx), free, fixed
        M = np.concatenate([_mass_diag(m)[:m["nf"]] for m in ms])
        dt = np.concatenate([np.full(m["nf"], d) for m, d in zip(ms, dts)])
        U, V, _ = _march(K, M, dt, 0.0, V0, np.zeros(free), np.zeros(case["steps"] + 1), case["steps"],
                         np.zeros(0, dtype=np.int64), 1, dev)
        return {"U": U, "V": V}
    m = _model(case, seed)
    if kind == "stiffness":
        return {"rowptr": None, "colval": None, "nzval": _csr_exact(m, case["block"], dev)}
    if kind == "request":
        return {"rowptr": None, "colval": None, "nzval": _csr_exact(m, "free", dev), "M": _mass_diag(m)[:m["nf"]]}
    if kind in ("explicit", "analysis"):
        V0, F, g, probes = _loads(case, m, seed)
        dt = _dt(m, seed)
        cd = 0.02 * 2 * (0.05 / dt) if case["damped"] else 0.0
        U, V, p = _march(_Operator(m, dev), _mass_diag(m)[:m["nf"]], dt, cd, V0, F, g, case["steps"], probes, 10, dev)
        return {"U": U, "V": V, "probes": p if probes.size else None}
    if kind == "stable_dt":
        K, M = _Operator(m, dev), _mass_diag(m)[:m["nf"]]
        Mt = torch.as_tensor(M, device=dev)
        v = torch.as_tensor(np.random.default_rng([seed, 16]).standard_normal(m["nf"]), device=dev)
        for _ in range(case["maxit"]):
            w = K(v)
            w = w / w.norm()
            v = w / Mt
            v = v / v.norm()
        return {"omega": float(torch.sqrt(torch.dot(v, K(v)) / torch.dot(v, Mt * v))), "M": M}
    if kind == "statics":
        u = np.random.default_rng([seed, 15]).normal(0.0, 1e-4, (m["xyz"].shape[0], 6))
        out, loc = _resultants_exact(m, u, dev)
        return {"F": _pressure_exact(m), "out": out, "loc": loc}
    raise ValueError(kind)
