"""Explicit loops on meshes with nodes that no element uses, their dofs free.
Such a node has an empty neighbour list and no mass: its own dofs come out as
not-a-number (as in the row products, whose rows are empty there), all others
bitwise as on the mesh without it.  Unused nodes last, first and between, alone and
several, below and above the step count from which loops run on patches."""
import numpy as np
import pytest

from flexshell import _lib, explicit, fe, femm as FM
from flexshell.material import MatDeforElastIso

pytestmark = pytest.mark.gpu

PRECISIONS = (_lib.FS_PREC_FP64, _lib.FS_PREC_MIXED, _lib.FS_PREC_MIXED_F32)


def _femm(ctx, xyz, conn, d):
    f = FM.make(conn, MatDeforElastIso(70e9, 0.33, 2700.0), thickness=0.02, ctx=ctx)
    f.associategeometry(xyz)
    f.stiffness(FM.SysmatAssemblerHIP(_lib.FS_BLOCK_FF), xyz, None, None, d)
    f.mass(FM.SysmatAssemblerHIP(_lib.FS_BLOCK_FF), xyz, d)
    return f


@pytest.mark.parametrize("nen, nx, ny", [(3, 5, 4), (4, 23, 19)])
@pytest.mark.parametrize("where", ["last", "first", "between", "several"])
def test_loop_with_unused_nodes(ctx, nen, nx, ny, where):
    print(f"[gpu] unused nodes {nen} {nx}x{ny} {where}", flush=True)
    xy, conn = (fe.T3block if nen == 3 else fe.Q4block)(0.1 * nx, 0.1 * ny, nx, ny)
    xyz = fe.xyz3(xy)
    xyz[:, 2] = 0.05 * np.sin(2.0 * xyz[:, 0])
    N = len(xyz)
    d = fe.DofField(N)
    d.setebc(np.nonzero(xy[:, 0] < 1e-9)[0], [1, 2, 3, 4, 5, 6])
    d.numberdofs()
    nf = d.nfreedofs
    # the same mesh with unused nodes before its nodes `at`
    at = {"last": [N], "first": [0], "between": [N // 2], "several": [0, 0, 7, N // 2, N, N]}[where]
    new = np.arange(N) + np.searchsorted(at, np.arange(N), side="right")
    Nu = N + len(at)
    used = np.zeros(Nu, dtype=bool)
    used[new] = True
    xyzu = np.full((Nu, 3), 3.0)
    xyzu[new] = xyz
    du = fe.DofField(Nu)
    du.setebc(new[np.nonzero(xy[:, 0] < 1e-9)[0]], [1, 2, 3, 4, 5, 6])
    du.numberdofs()
    nu = du.nfreedofs
    assert nu == nf + 6 * len(at)
    rows = du.dofnums[used]
    rows = np.sort(rows[rows < nu])  # the used nodes' free dofs, in their order
    f, fu = _femm(ctx, xyz, conn, d), _femm(ctx, xyzu, new[conn], du)
    rng = np.random.default_rng(3)
    dt = 0.8 * explicit.stable_dt(explicit.omega_max(f, rng.standard_normal(nf), 100))
    U0, V0, F = rng.normal(0, 1e-6, nf), rng.normal(0, 1e-3, nf), rng.normal(0, 1.0, nf)
    probes = np.array([0, nf // 2, nf - 1])

    def wide(v):
        out = np.zeros(nu)
        out[rows] = v
        return out

    for prec in PRECISIONS:
        for nsteps in (20, 120):
            g = np.where(np.arange(nsteps + 1) < 40, np.cos(0.1 * np.arange(nsteps + 1)), 0.0)
            a = explicit.run(f._model, 30.0, U0, V0, dt, nsteps, F, g, probes, 7, prec)
            b = explicit.run(fu._model, 30.0, wide(U0), wide(V0), dt, nsteps, wide(F), g, rows[probes], 7, prec)
            assert np.all(np.isfinite(a["U"])) and np.any(a["U"])
            for key in ("U", "V"):
                assert np.array_equal(a[key], b[key][rows]), (prec, nsteps, key)
                assert np.all(np.isnan(np.delete(b[key], rows))), (prec, nsteps, key)
            assert np.array_equal(a["probes"], b["probes"]), (prec, nsteps)
    f._model.close()
    fu._model.close()
