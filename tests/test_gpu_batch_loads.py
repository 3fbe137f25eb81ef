"""Batches stepped on patches with a load history, damping and a time step per model,
and probes: both element families, the three precisions, more patches than one
launch takes, in one launch per set of models and step by step.  Each model bitwise as
alone; against the oracle's loop 1e-10 relative in FP64 and 1e-9 in the mixed
precisions (values to a relative 2^-39: over 120 steps at omega dt <= 2 a phase error
of 4.4e-10)."""
import numpy as np
import pytest

from flexshell import _lib, batch as FB, explicit, fe, femm as FM
from flexshell.material import MatDeforElastIso
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _model(nen, nx, ny, k):
    xy, conn = (fe.T3block if nen == 3 else fe.Q4block)(0.1 * nx, 0.1 * ny, nx, ny)
    xyz = fe.xyz3(xy)
    xyz[:, 2] = 0.05 * np.sin(2.0 * xyz[:, 0] + k)
    d = fe.DofField(len(xyz))
    d.setebc(np.nonzero(xy[:, 0] < 1e-9)[0], [1, 2, 3, 4, 5, 6] if k % 2 else [1, 2, 3])
    d.numberdofs()
    return dict(xyz=xyz, conn=conn, dchi=d, material=MatDeforElastIso((1 + k) * 3e10, 0.3, 2000.0 + 100 * k),
                t=0.02 + 0.001 * k)


@pytest.mark.parametrize("nen", [3, 4])
@pytest.mark.parametrize("prec", [_lib.FS_PREC_FP64, _lib.FS_PREC_MIXED, _lib.FS_PREC_MIXED_F32])
def test_loaded_damped_batch(ctx, nen, prec):
    print(f"[gpu] loaded batch nen {nen} precision {prec}", flush=True)
    sizes = [(60, 50), (7, 6), (61, 47), (55, 55), (2, 2), (70, 44), (40, 80), (58, 52), (33, 97)]
    models = [_model(nen, nx, ny, k) for k, (nx, ny) in enumerate(sizes)]
    nm, nsteps, stride = len(models), 120, 7
    assert sum(-(-len(m["xyz"]) // 42) for m in models) > 512
    b = FB.ShellBatch(models, ctx=ctx)
    b.assemble_device()
    b.mass()
    n = b.nfree
    rng = np.random.default_rng(9)
    U0, V0, F = rng.normal(0, 1e-6, n), rng.normal(0, 1e-3, n), rng.normal(0, 1.0, n)
    cd = np.array([0.0, 40.0, 25.0, 0.0, 60.0, 10.0, 0.0, 35.0, 5.0])
    i = np.arange(nsteps + 1)[:, None]
    g = np.cos(0.1 * i * (1 + np.arange(nm) % 4)) * (i < 30 + 10 * np.arange(nm))
    probes = np.sort(rng.choice(n, 60, replace=False))
    K, M, dts = [], [], []
    for m in models:
        f = FM.make(m["conn"], m["material"], thickness=m["t"], ctx=ctx)
        f.associategeometry(m["xyz"])
        nf = m["dchi"].nfreedofs
        K.append(f.stiffness(FM.SysmatAssemblerFFBlock(nf), m["xyz"], None, None, m["dchi"]))
        M.append(f.mass(FM.SysmatAssemblerFFBlock(FM.SysmatAssemblerSparseDiag(), nf, nf), m["xyz"],
                        m["dchi"]).diagonal())
        m["femm"] = f
        dts.append(0.8 * explicit.stable_dt(explicit.omega_max(f, rng.standard_normal(nf), 150)))
    dts = np.array(dts)

    def run(graph):
        return b.explicit(dts, cd, U0, V0, F, g, nsteps, use_graph=graph, probe_dofs=probes, probe_stride=stride,
                          precision=prec)

    try:
        ctx.set_cd_loop(-1)
        step = run(False)
        assert b.model.cd_form() == _lib.FS_CD_PATCHES
        graph = run(True)
    finally:
        ctx.set_cd_loop(0)
    loop = run(False)
    assert b.model.cd_form() == _lib.FS_CD_ONE_LAUNCH
    for other in (graph, loop, run(True), run(True)):
        for key in ("U", "V", "probes"):
            assert np.array_equal(step[key], other[key]), key
    tol = 1e-10 if prec == _lib.FS_PREC_FP64 else 1e-9
    for k, m in enumerate(models):
        sl = b.model_slice(k)
        mine = np.nonzero((probes >= sl.start) & (probes < sl.stop))[0]
        args = (F[sl], g[:, k])
        r = explicit.run(m["femm"]._model, cd[k], U0[sl], V0[sl], dts[k], nsteps, *args, probes[mine] - sl.start, stride,
                         prec)
        m["femm"]._model.close()
        assert np.array_equal(r["U"], step["U"][sl]) and np.array_equal(r["V"], step["V"][sl]), k
        assert np.array_equal(r["probes"], step["probes"][:, mine]), k
        Uo, Vo, po = O.cd_loop(K[k], M[k], cd[k], dts[k], nsteps, *args, U0[sl], V0[sl], probes[mine] - sl.start)
        assert np.linalg.norm(r["U"] - Uo) <= tol * np.linalg.norm(Uo), k
        assert np.linalg.norm(r["V"] - Vo) <= tol * np.linalg.norm(Vo), k
        if len(mine):
            assert np.linalg.norm(r["probes"] - po[::stride]) <= tol * np.linalg.norm(po), k
    b.close()
