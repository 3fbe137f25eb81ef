"""Probes of the explicit loop: few, many, all dofs, the same dof twice (the later
probe records it), in every form of the loop; each record against the
displacement that a loop of that many steps ends with.  With as many probes as
dofs the call takes at most a few times what it takes without probes, less the
copy of the records."""
import time

import numpy as np
import pytest

from flexshell import _lib, explicit, fe, femm as FM
from flexshell.material import MatDeforElastIso

pytestmark = pytest.mark.gpu


def _model(ctx, nx, ny):
    xy, conn = fe.Q4block(0.1 * nx, 0.1 * ny, nx, ny)
    xyz = fe.xyz3(xy)
    d = fe.DofField(len(xyz))
    d.setebc(np.nonzero(xy[:, 0] < 1e-9)[0], [1, 2, 3])
    d.numberdofs()
    f = FM.make(conn, MatDeforElastIso(70e9, 0.33, 2700.0), thickness=0.02, ctx=ctx)
    f.associategeometry(xyz)
    f.stiffness(FM.SysmatAssemblerHIP(_lib.FS_BLOCK_FF), xyz, None, None, d)
    f.mass(FM.SysmatAssemblerHIP(_lib.FS_BLOCK_FF), xyz, d)
    return f, d.nfreedofs


@pytest.mark.parametrize("nsteps", [30, 120])
@pytest.mark.parametrize("prec", [_lib.FS_PREC_FP64, _lib.FS_PREC_MIXED_F32])
def test_probe_records(ctx, nsteps, prec):
    print(f"[gpu] probes {nsteps} steps precision {prec}", flush=True)
    f, n = _model(ctx, 13, 9)
    rng = np.random.default_rng(1)
    z, V0 = np.zeros(n), rng.normal(0, 1e-3, n)
    dt = 0.5 * explicit.stable_dt(explicit.omega_max(f, rng.standard_normal(n), 100))

    def run(steps, probes=(), stride=1):
        return explicit.run(f._model, 0.0, z, V0, dt, steps, z, np.zeros(steps + 1), probes, stride, prec)

    end = run(nsteps)["U"]
    for probes in (np.array([n - 1]), rng.permutation(n)[:257], rng.permutation(n)):
        r = run(nsteps, probes, nsteps)
        assert np.array_equal(r["U"], end) and np.array_equal(r["probes"][0], z[probes])
        # the record of a step is U as that step starts from it: of the last one, U_nsteps
        assert np.array_equal(r["probes"][1], end[probes])
    twice = np.array([3, 0, 3, n - 1, 0, 3])
    r = run(nsteps, twice, 10)
    single = run(nsteps, np.array([0, 3, n - 1]), 10)["probes"]
    assert np.array_equal(r["probes"][1:, [4, 5, 3]], single[1:])
    f._model.close()


def test_probes_on_all_dofs_cost_their_records(ctx):
    print("[gpu] probes on all dofs", flush=True)
    f, n = _model(ctx, 300, 200)
    z = np.zeros(n)
    V0 = np.random.default_rng(0).normal(0, 1e-3, n)

    def ms(probes):
        best = np.inf
        for _ in range(5):
            t = time.perf_counter()
            explicit.run(f._model, 0.0, z, V0, 1e-8, 20, z, np.zeros(21), probes, 20)
            best = min(best, (time.perf_counter() - t) * 1e3)
        return best

    without, alldofs = ms(()), ms(np.arange(n))
    # two records of n values, their upload and their copy: 1 to 3 ms here
    assert alldofs <= 3.0 * without + 6.0, (without, alldofs)
    f._model.close()
