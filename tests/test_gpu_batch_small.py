"""Batches of models smaller than a patch, which share patches: every model bitwise
as alone (where its patch is its own), in the three precisions, step by step and in
one launch; sizes at and around the patch's 42 nodes, a hub whose neighbours fill a
patch's partial slots, fixed nodes only in part, larger models between.  And a
batch of very small models is stepped no slower than with the row products."""
import numpy as np
import pytest

from flexshell import _lib, batch as FB, explicit, fe, femm as FM
from flexshell.material import MatDeforElastIso

pytestmark = pytest.mark.gpu

MAT = MatDeforElastIso(70e9, 0.33, 2700.0)


def _plate(nx, ny, clamp):
    xy, conn = fe.T3block(0.1 * nx, 0.1 * ny, nx, ny)
    xyz = fe.xyz3(xy)
    xyz[:, 2] = 0.05 * np.sin(2.0 * xyz[:, 0])
    d = fe.DofField(len(xyz))
    if clamp:
        d.setebc(np.nonzero(xy[:, 0] < 1e-9)[0], clamp)
    d.numberdofs()
    return dict(xyz=xyz, conn=conn, dchi=d, material=MAT, t=0.02)


def _fan(m):
    a = 2 * np.pi * np.arange(m) / m
    xyz = np.vstack([[0.0, 0.0, 0.0], np.column_stack([np.cos(a), np.sin(a), 0 * a])])
    conn = np.column_stack([np.zeros(m, dtype=np.int64), 1 + np.arange(m), 1 + (np.arange(m) + 1) % m])
    d = fe.DofField(m + 1)
    d.setebc([1, 2], [1, 2, 3, 4, 5, 6])
    d.numberdofs()
    return dict(xyz=xyz, conn=conn, dchi=d, material=MAT, t=0.02)


ALL = [1, 2, 3, 4, 5, 6]


def _models():
    small = [_plate(1, 1, None), _plate(2, 2, [1, 2, 3]), _plate(1, 2, ALL), _plate(5, 6, None),  # 4, 9, 4, 42
             _plate(1, 1, ALL), _plate(20, 1, ALL), _plate(20, 1, None), _plate(1, 20, [2, 4]),  # 2, 40, 42, 42
             _plate(42, 1, ALL), _fan(60), _plate(13, 9, ALL), _plate(1, 1, None), _plate(2, 1, [3]), _fan(9)]
    return small + [_plate(2, 2, [1, 2, 3]) for _ in range(40)]


@pytest.mark.parametrize("prec", [_lib.FS_PREC_FP64, _lib.FS_PREC_MIXED, _lib.FS_PREC_MIXED_F32])
def test_small_models_as_alone(ctx, prec):
    print(f"[gpu] batch of small models, precision {prec}", flush=True)
    models = _models()
    nm, nsteps = len(models), 110
    rng = np.random.default_rng(5)
    b = FB.ShellBatch(models, ctx=ctx)
    b.assemble_device()
    b.mass()
    n = b.nfree
    U0, V0, F = rng.normal(0, 1e-6, n), rng.normal(0, 1e-3, n), rng.normal(0, 1.0, n)
    cd = np.where(np.arange(nm) % 3 == 0, 30.0, 0.0)
    g = np.cos(0.1 * np.arange(nsteps + 1)[:, None] * (1 + np.arange(nm) % 5)) * (np.arange(nsteps + 1) < 70)[:, None]
    probes = np.sort(rng.choice(n, 40, replace=False))
    # a step of the smallest elements' order, far below every model's limit
    dts = np.where(np.arange(nm) % 2 == 0, 4e-8, 3e-8)
    try:
        ctx.set_cd_loop(-1)
        step = b.explicit(dts, cd, U0, V0, F, g, nsteps, use_graph=False, probe_dofs=probes, probe_stride=9,
                          precision=prec)
    finally:
        ctx.set_cd_loop(0)
    loop = b.explicit(dts, cd, U0, V0, F, g, nsteps, use_graph=False, probe_dofs=probes, probe_stride=9, precision=prec)
    assert np.all(np.isfinite(step["U"])) and np.any(step["U"])
    for key in ("U", "V", "probes"):
        assert np.array_equal(step[key], loop[key]), key
    for k in [*range(16), nm - 1]:
        m, sl = models[k], b.model_slice(k)
        f = FM.make(m["conn"], MAT, thickness=0.02, ctx=ctx)
        f.associategeometry(m["xyz"])
        f.stiffness(FM.SysmatAssemblerHIP(_lib.FS_BLOCK_FF), m["xyz"], None, None, m["dchi"])
        f.mass(FM.SysmatAssemblerHIP(_lib.FS_BLOCK_FF), m["xyz"], m["dchi"])
        mine = np.nonzero((probes >= sl.start) & (probes < sl.stop))[0]
        r = explicit.run(f._model, cd[k], U0[sl], V0[sl], dts[k], nsteps, F[sl], g[:, k], probes[mine] - sl.start, 9,
                         prec)
        f._model.close()
        assert np.array_equal(r["U"], step["U"][sl]) and np.array_equal(r["V"], step["V"][sl]), k
        assert np.array_equal(r["probes"], step["probes"][:, mine]), k
    b.close()


def test_tiny_models_step_time(ctx):
    print("[gpu] batch of tiny models, time", flush=True)
    nm, nsteps = 4000, 300
    b = FB.ShellBatch([_plate(1, 1, None)] * nm, ctx=ctx)
    b.assemble_device()
    b.mass()
    z, V0 = np.zeros(b.nfree), np.random.default_rng(0).normal(0, 1e-3, b.nfree)

    def ms():
        return min(b.explicit(np.full(nm, 1e-8), np.zeros(nm), z, V0, z, np.zeros((nsteps + 1, nm)), nsteps,
                              use_graph=False)["ms"] for _ in range(4))

    patches = ms()
    try:
        ctx.set_cd_lanes(8, 4)
        rows = ms()
    finally:
        ctx.set_cd_lanes(8)
    assert patches <= 1.1 * rows, (patches, rows)
    b.close()
