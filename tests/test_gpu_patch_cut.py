"""Patches cut by kernels and by the host are the same.  A mesh of at least 2048
nodes is cut by kernels alone, and by the host where a component with a hub stands
beside it; a component's results depend on its own patches only, so that they are
bitwise the same both ways.  Regular grids (ties along both axes), a jittered one,
a strip, sizes just past the limit and past a 1024-lane level (4096 nodes)."""
import numpy as np
import pytest

from test_gpu_patch_step import _fan
from flexshell import explicit, fe, femm as FM
from flexshell.material import MatDeforElastIso

pytestmark = pytest.mark.gpu


def _run(ctx, nen, xyz, conn, clamp, U0, V0, dt):
    d = fe.DofField(len(xyz))
    d.setebc(clamp, [1, 2, 3, 4, 5, 6])
    d.numberdofs()
    f = FM.make(conn, MatDeforElastIso(70e9, 0.33, 2700.0), thickness=0.02, ctx=ctx)
    f.associategeometry(xyz)
    f.stiffness(FM.SysmatAssemblerHIP(), xyz, None, None, d)
    f.mass(FM.SysmatAssemblerHIP(), xyz, d)
    nf = d.nfreedofs
    z = np.zeros(nf)
    u, v = z.copy(), z.copy()
    u[:len(U0)], v[:len(V0)] = U0, V0
    if dt is None:
        dt = 0.5 * explicit.stable_dt(explicit.omega_max(f, np.random.default_rng(1).standard_normal(nf), 100))
    r = explicit.run(f._model, 0.0, u, v, dt, 100, z, np.zeros(101))
    f._model.close()
    return r["U"], r["V"], dt


@pytest.mark.parametrize("nx, ny, jitter", [(50, 40, 0.0), (70, 64, 0.0), (90, 81, 0.2), (1400, 1, 0.0)])
def test_kernel_cuts_match_host_cuts(ctx, nx, ny, jitter):
    print(f"[gpu] patch cuts {nx}x{ny} jitter {jitter}", flush=True)
    xy, conn = fe.T3block(0.1 * nx, 0.1 * ny, nx, ny)
    rng = np.random.default_rng(nx)
    xyz = fe.xyz3(xy + 0.1 * jitter * rng.uniform(-1, 1, xy.shape))
    xyz[:, 2] = 0.05 * np.sin(2.0 * xyz[:, 0])
    clamp = np.nonzero(xy[:, 0] < 1e-9)[0]
    n = 6 * (len(xyz) - len(clamp))
    U0, V0 = rng.normal(0, 1e-6, n), rng.normal(0, 1e-3, n)
    U, V, dt = _run(ctx, 3, xyz, conn, clamp, U0, V0, None)
    _, xh, ch, _ = _fan(40)
    Uh, Vh, _ = _run(ctx, 3, np.vstack([xyz, xh + [0.0, 0.0, 50.0]]), np.vstack([conn, ch + len(xyz)]),
                     np.concatenate([clamp, len(xyz) + np.arange(1, 4)]), U0, V0, dt)
    assert np.all(np.isfinite(U)) and np.any(U)
    assert np.array_equal(Uh[:n], U) and np.array_equal(Vh[:n], V)
