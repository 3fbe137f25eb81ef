"""The form that an explicit loop takes, as the model reports it, where the other
tests compare the forms' results: one launch where the mesh is small and there is
room, step by step where that is asked for, where the mesh is large or where loops
at the same time have no room, again step by step where a wait ran out, and the
row products for short loops, chosen row forms and hubs past a patch."""
import threading

import numpy as np
import pytest

import test_gpu_patch_step as PS
from flexshell import _lib, batch as FB, explicit, fe, femm as FM
from flexshell.material import MatDeforElastIso

pytestmark = pytest.mark.gpu

ROWS, PATCHES, ONE, RESTARTED = _lib.FS_CD_ROWS, _lib.FS_CD_PATCHES, _lib.FS_CD_ONE_LAUNCH, _lib.FS_CD_RESTARTED
PRECISIONS = (_lib.FS_PREC_FP64, _lib.FS_PREC_MIXED, _lib.FS_PREC_MIXED_F32)


def _femm(ctx, mesh):
    nen, xyz, conn, d = mesh
    f = FM.make(conn, MatDeforElastIso(70e9, 0.33, 2700.0), thickness=0.02, ctx=ctx)
    f.associategeometry(xyz)
    f.stiffness(FM.SysmatAssemblerHIP(_lib.FS_BLOCK_FF), xyz, None, None, d)
    f.mass(FM.SysmatAssemblerHIP(_lib.FS_BLOCK_FF), xyz, d)
    V0 = np.random.default_rng(1).normal(0, 1e-3, d.nfreedofs)
    z = np.zeros(d.nfreedofs)

    def run(nsteps=100, prec=_lib.FS_PREC_FP64, graph=False):
        explicit.run(f._model, 0.0, z, V0, 1e-8, nsteps, z, np.zeros(nsteps + 1), (), 1, prec, use_graph=graph)
        return f._model.cd_form()

    return f, run


@pytest.mark.parametrize("nen, nx, ny", [(4, 3, 2), (4, 97, 61), (3, 140, 70)])
def test_one_launch_is_taken(ctx, nen, nx, ny):
    print(f"[gpu] loop form {nen} {nx}x{ny}", flush=True)
    f, run = _femm(ctx, PS._grid(nen, nx, ny, "partial"))
    assert f._model.cd_form() == -1
    for prec in PRECISIONS:
        for graph in (False, True, True):
            assert run(100, prec, graph) == ONE
    assert run(99) == ROWS
    try:
        ctx.set_cd_loop(-1)
        assert run() == PATCHES and run(graph=True) == PATCHES
        ctx.set_cd_lanes(0)
        assert run() == ROWS and run(100, _lib.FS_PREC_MIXED_F32) == PATCHES
        ctx.set_cd_lanes(8)
        ctx.set_cd_loop(1)
        if nx > 3:  # a limit of one poll: a wait runs out, and the context stays off the form
            assert run() == RESTARTED and run() == PATCHES
        else:  # one patch waits for none
            assert run() == ONE
    finally:
        ctx.set_cd_lanes(8)
        ctx.set_cd_loop(0)
    assert run() == ONE
    f._model.close()


def test_other_forms(ctx):
    print("[gpu] loop forms of other meshes", flush=True)
    for mesh, form in ((PS._grid(4, 230, 200), PATCHES),  # more patches than one launch takes
                       (PS._fan(40), ONE), (PS._fan(300), PATCHES), (PS._fan(1100), ROWS), (PS._two(), ONE)):
        f, run = _femm(ctx, mesh)
        assert run() == form, len(mesh[1])
        f._model.close()
    # the meshes whose cuts are compared elsewhere, alone and with a hub beside them
    _, xh, ch, _ = PS._fan(40)
    for nx, ny in ((50, 40), (70, 64), (90, 81), (1400, 1)):
        xy, conn = fe.T3block(0.1 * nx, 0.1 * ny, nx, ny)
        xyz = fe.xyz3(xy)
        for x, c in ((xyz, conn), (np.vstack([xyz, xh + [0.0, 0.0, 50.0]]), np.vstack([conn, ch + len(xyz)]))):
            d = fe.DofField(len(x))
            d.setebc(np.nonzero(xy[:, 0] < 1e-9)[0], [1, 2, 3, 4, 5, 6])
            d.numberdofs()
            f, run = _femm(ctx, (3, x, c, d))
            assert run() in (PATCHES, ONE), (nx, ny, len(x))
            f._model.close()


def test_loops_at_the_same_time(ctx):
    """Four contexts with 245 patches each, of which two fit the device together."""
    print("[gpu] loop forms of four contexts", flush=True)
    jobs = [_femm(_lib.Context(ctx.device), PS._grid(3, 140, 70)) for _ in range(4)]
    start = threading.Barrier(4)
    got = [[] for _ in jobs]

    def work(k):
        start.wait()
        got[k].extend(jobs[k][1](3000) for _ in range(4))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    forms = sum(got, [])
    assert len(forms) == 16 and ONE in forms and set(forms) <= {PATCHES, ONE}, got
    assert all(run() == ONE for _, run in jobs)  # none has left the form
    for f, _ in jobs:
        f._model.close()


def test_batch_with_a_hub_past_a_patch(ctx):
    """The row products for the whole batch: a model beside the hub equals itself alone
    (on patches) up to the order of addition, 1e-12 relative as between the forms."""
    print("[gpu] batch with a hub", flush=True)
    models = [dict(xyz=xyz, conn=conn, dchi=d, material=MatDeforElastIso(70e9, 0.33, 2700.0), t=0.02)
              for _, xyz, conn, d in (PS._grid(3, 17, 13), PS._fan(1100))]
    b = FB.ShellBatch(models, ctx=ctx)
    b.assemble_device()
    b.mass()
    V0, z = np.random.default_rng(6).normal(0, 1e-3, b.nfree), np.zeros(b.nfree)
    r = b.explicit([1e-8] * 2, [0.0] * 2, z, V0, z, np.zeros((121, 2)), 120, use_graph=False)
    assert b.model.cd_form() == ROWS
    m, sl = models[0], b.model_slice(0)
    f, run = _femm(ctx, (3, m["xyz"], m["conn"], m["dchi"]))
    a = explicit.run(f._model, 0.0, z[sl], V0[sl], 1e-8, 120, z[sl], np.zeros(121))
    assert f._model.cd_form() == ONE
    for key in ("U", "V"):
        assert np.linalg.norm(a[key] - r[key][sl]) <= 1e-12 * np.linalg.norm(a[key]), key
    f._model.close()
    b.close()
