"""The explicit step on the patch form of K (the default of loops of 100
steps or more) against the row products and the oracle.

Both forms add the same products in different orders: 1e-12 relative between
them over 120 steps at 0.8 of the stable dt (the bound of the row forms among
themselves), 1e-10 against the oracle's loop.  The mixed precisions hold
values to a relative 2^-39: over n steps at omega dt <= 2 a phase error of 2 n
2^-39, 4.4e-10 for 120 steps, bounded by 1e-9 against the oracle.  Meshes at the edges of the
plan: one node with free dofs, one and two patches (42 and 43 nodes), a hub
whose patch has more blocks than the workgroup has lanes, a hub of more
neighbours than a patch takes (row products throughout), two components,
partly fixed nodes, a permuted numbering."""
import threading

import numpy as np
import pytest

from flexshell import _lib, explicit, fe, femm as FM
from flexshell.material import MatDeforElastIso
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _grid(nen, nx, ny, clamp="left", perm=False):
    xy, conn = (fe.T3block if nen == 3 else fe.Q4block)(0.1 * nx, 0.1 * ny, nx, ny)
    xyz = fe.xyz3(xy)
    xyz[:, 2] = 0.05 * np.sin(2.0 * xyz[:, 0])
    d = fe.DofField(xyz.shape[0])
    left = xy[:, 0] < 1e-9
    if clamp == "left":
        d.setebc(np.nonzero(left)[0], [1, 2, 3, 4, 5, 6])
    elif clamp == "partial":
        d.setebc(np.nonzero(left)[0], [1, 2, 3])
        d.setebc(np.nonzero(xy[:, 1] < 1e-9)[0], [3, 5])
    else:
        d.setebc(np.arange(1, xyz.shape[0]), [1, 2, 3, 4, 5, 6])
    d.numberdofs(perm=np.random.default_rng(5).permutation(xyz.shape[0]) if perm else None)
    return nen, xyz, conn, d


def _fan(m):
    a = 2 * np.pi * np.arange(m) / m
    xyz = np.vstack([[0.0, 0.0, 0.0], np.column_stack([np.cos(a), np.sin(a), 0 * a])])
    conn = np.column_stack([np.zeros(m, dtype=np.int64), 1 + np.arange(m), 1 + (np.arange(m) + 1) % m])
    d = fe.DofField(m + 1)
    d.setebc([1, 2, 3], [1, 2, 3, 4, 5, 6])
    d.numberdofs()
    return 3, xyz, conn, d


def _two():
    _, x1, c1, _ = _grid(4, 7, 6)
    _, x2, c2, _ = _grid(4, 3, 11)
    xyz = np.vstack([x1, x2 + [5.0, 0.0, 0.0]])
    conn = np.vstack([c1, c2 + len(x1)])
    d = fe.DofField(len(xyz))
    d.setebc([0, 1, 2, len(x1), len(x1) + 1], [1, 2, 3, 4, 5, 6])
    d.numberdofs()
    return 4, xyz, conn, d


MESHES = {
    "one_node": lambda: _grid(4, 3, 3, "all_but_one"),
    "q4_42": lambda: _grid(4, 6, 6),               # 42 of 49 nodes have free dofs
    "q4_43": lambda: _grid(4, 1, 42),
    "t3_43": lambda: _grid(3, 1, 42),
    "t3_perm": lambda: _grid(3, 17, 13, perm=True),
    "q4_partial": lambda: _grid(4, 23, 9, "partial"),
    "hub_300": lambda: _fan(300),
    "hub_1100": lambda: _fan(1100),
    "two": _two,
}


@pytest.mark.parametrize("nen,nx,ny", [(4, 3, 2), (3, 9, 7), (4, 97, 61), (3, 140, 70)],
                         ids=["one_patch", "t3", "q4_146_patches", "t3_245_patches"])
@pytest.mark.parametrize("prec", [_lib.FS_PREC_FP64, _lib.FS_PREC_MIXED_F32], ids=["fp64", "f32"])
def test_loop_in_one_launch(ctx, nen, nx, ny, prec):
    """The one-launch loop gives bitwise what the same steps give one by one,
    in a graph too, with odd and even step counts, and where its waits run out
    (a limit of one poll), in which case the call runs step by step."""
    print(f"[gpu] loop in one launch {nen} {nx}x{ny} precision {prec}", flush=True)
    _, xyz, conn, d = _grid(nen, nx, ny, "partial")
    f = FM.make(conn, MatDeforElastIso(70e9, 0.33, 2700.0), thickness=0.02, ctx=ctx)
    f.associategeometry(xyz)
    nf = d.nfreedofs
    f.stiffness(FM.SysmatAssemblerHIP(), xyz, None, None, d)
    f.mass(FM.SysmatAssemblerHIP(), xyz, d)
    rng = np.random.default_rng(3)
    dt = 0.8 * explicit.stable_dt(explicit.omega_max(f, rng.standard_normal(nf), 200))
    U0, V0, F = rng.normal(0, 1e-6, nf), rng.normal(0, 1e-3, nf), rng.normal(0, 1.0, nf)
    probes = rng.choice(nf, 5, replace=False)

    def run(polls, nsteps, cdamp, graph=False):
        ctx.set_cd_loop(polls)
        try:
            g = np.where(np.arange(nsteps + 1) % 50 < 20, np.cos(0.1 * np.arange(nsteps + 1)), 0.0)
            return explicit.run(f._model, cdamp, U0, V0, dt, nsteps, F, g, probes, 7, prec, use_graph=graph)
        finally:
            ctx.set_cd_loop(0)

    for nsteps, cdamp in ((100, 0.0), (301, 40.0)):
        ref = run(-1, nsteps, cdamp)
        for polls, graph in ((0, False), (0, True), (0, True), (1, False), (0, False)):
            r = run(polls, nsteps, cdamp, graph)
            for key in ("U", "V", "probes"):
                assert np.array_equal(r[key], ref[key]), (nsteps, polls, graph, key)
    f._model.close()


def test_loops_at_the_same_time(ctx):
    """Contexts whose loops together have more patches than the device has
    places for: some run step by step meanwhile, all give what they give alone."""
    print("[gpu] loops of four contexts", flush=True)
    jobs = []
    for k in range(4):
        c = _lib.Context(ctx.device)
        _, xyz, conn, d = _grid(3, 140, 70 - k)
        f = FM.make(conn, MatDeforElastIso(70e9, 0.33, 2700.0), thickness=0.02, ctx=c)
        f.associategeometry(xyz)
        f.stiffness(FM.SysmatAssemblerHIP(), xyz, None, None, d)
        f.mass(FM.SysmatAssemblerHIP(), xyz, d)
        nf = d.nfreedofs
        dt = 0.8 * explicit.stable_dt(explicit.omega_max(f, np.random.default_rng(k).standard_normal(nf), 200))
        V0, z = np.random.default_rng(k).normal(0, 1e-3, nf), np.zeros(nf)
        jobs.append((f, lambda m=f._model, z=z, V0=V0, dt=dt: explicit.run(m, 0.0, z, V0, dt, 2000, z, np.zeros(2001))))
    alone = [run() for _, run in jobs]
    got = [[] for _ in jobs]
    threads = [threading.Thread(target=lambda k=k: got[k].extend(jobs[k][1]() for _ in range(5))) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, rs in zip(alone, got):
        assert len(rs) == 5
        for r in rs:
            assert np.array_equal(a["U"], r["U"]) and np.array_equal(a["V"], r["V"])
    for f, _ in jobs:
        f._model.close()


@pytest.mark.parametrize("name", list(MESHES))
@pytest.mark.parametrize("cdamp,form", [(0.0, 0), (50.0, 1)], ids=["undamped", "damped_average_k"])
def test_patch_step(ctx, name, cdamp, form):
    print(f"[gpu] patch step {name} {cdamp}", flush=True)
    nen, xyz, conn, d = MESHES[name]()
    f = FM.make(conn, MatDeforElastIso(70e9, 0.33, 2700.0), thickness=0.02, ctx=ctx)
    f.transv_shear_formulation = form if nen == 3 else 0
    f.associategeometry(xyz)
    nf = d.nfreedofs
    K = f.stiffness(FM.SysmatAssemblerFFBlock(nf), xyz, None, None, d)
    M = f.mass(FM.SysmatAssemblerFFBlock(FM.SysmatAssemblerSparseDiag(), nf, nf), xyz, d).diagonal()
    rng = np.random.default_rng(7)
    U0, V0, F = rng.normal(0, 1e-6, nf), rng.normal(0, 1e-3, nf), rng.normal(0, 1.0, nf)
    dt = 0.8 * explicit.stable_dt(O.pwr(K, M, rng.standard_normal(nf), 200))
    nsteps = 120
    g = np.where(np.arange(nsteps + 1) < 40, np.cos(0.1 * np.arange(nsteps + 1)), 0.0)
    probes = np.array([nf - 1, 0, nf // 2])
    Uo, Vo, po = O.cd_loop(K, M, cdamp, dt, nsteps, F, g, U0, V0, probes)
    r = explicit.run(f._model, cdamp, U0, V0, dt, nsteps, F, g, probes, 7)
    again = explicit.run(f._model, cdamp, U0, V0, dt, nsteps, F, g, probes, 7, use_graph=True)
    try:
        ctx.set_cd_lanes(0)
        rows = explicit.run(f._model, cdamp, U0, V0, dt, nsteps, F, g, probes, 7)
    finally:
        ctx.set_cd_lanes(8)
    for key, ref in (("U", Uo), ("V", Vo)):
        assert np.array_equal(r[key], again[key])
        assert np.linalg.norm(r[key] - rows[key]) <= 1e-12 * np.linalg.norm(rows[key]), key
        assert np.linalg.norm(r[key] - ref) <= 1e-10 * np.linalg.norm(ref), key
    assert np.linalg.norm(r["probes"] - po[::7]) <= 1e-10 * np.linalg.norm(po)
    # the mixed precisions on the same plan, also after one another
    for prec in (_lib.FS_PREC_MIXED, _lib.FS_PREC_MIXED_F32, _lib.FS_PREC_MIXED):
        q = explicit.run(f._model, cdamp, U0, V0, dt, nsteps, F, g, probes, 7, precision=prec)
        for key, ref in (("U", Uo), ("V", Vo)):
            assert np.linalg.norm(q[key] - ref) <= 1e-9 * np.linalg.norm(ref), (prec, key)
    back = explicit.run(f._model, cdamp, U0, V0, dt, nsteps, F, g, probes, 7)
    assert np.array_equal(r["U"], back["U"]) and np.array_equal(r["V"], back["V"])
    # new values behind the same plan
    f.thickness = 0.03
    f.stiffness(FM.SysmatAssemblerHIP(_lib.FS_BLOCK_FF), xyz, None, None, d)
    a = explicit.run(f._model, cdamp, U0, V0, 0.5 * dt, nsteps, F, g)
    try:
        ctx.set_cd_lanes(0)
        b = explicit.run(f._model, cdamp, U0, V0, 0.5 * dt, nsteps, F, g)
    finally:
        ctx.set_cd_lanes(8)
    assert np.linalg.norm(a["U"] - b["U"]) <= 1e-12 * np.linalg.norm(b["U"])
    f._model.close()
