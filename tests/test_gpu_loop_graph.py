"""Graphs of the one-launch loop and new equation numbers: two components, each a
launch of its own, whose patches move from one to the other with the supports while
all totals stay.  A graph of the old launches would split a component over two, whose
waits on each other run out."""
import numpy as np
import pytest

import test_gpu_patch_step as PS
from flexshell import _lib, explicit, fe, femm as FM
from flexshell.material import MatDeforElastIso

pytestmark = pytest.mark.gpu


def test_graph_follows_the_components(ctx):
    print("[gpu] loop graph, moved supports", flush=True)
    _, x, c, _ = PS._grid(3, 150, 80)
    N = len(x)
    xyz, conn = np.vstack([x, x + [0.0, 0.0, 40.0]]), np.vstack([c, c + N])
    f = FM.make(conn, MatDeforElastIso(70e9, 0.33, 2700.0), thickness=0.02, ctx=ctx)
    f.associategeometry(xyz)
    V0 = None
    for turn in range(4):
        d = fe.DofField(2 * N)
        fixed = np.arange(81 * 10)  # the first rows of nodes along one edge
        d.setebc(fixed + (N if turn % 2 else 0), [1, 2, 3, 4, 5, 6])
        d.numberdofs()
        nf = d.nfreedofs
        if V0 is None:
            V0, n0 = np.random.default_rng(2).normal(0, 1e-3, nf), nf
        assert nf == n0
        f.stiffness(FM.SysmatAssemblerHIP(_lib.FS_BLOCK_FF), xyz, None, None, d)
        f.mass(FM.SysmatAssemblerHIP(_lib.FS_BLOCK_FF), xyz, d)
        z = np.zeros(nf)

        def run(graph):
            r = explicit.run(f._model, 0.0, z, V0, 1e-8, 120, z, np.zeros(121), use_graph=graph)
            assert f._model.cd_form() == _lib.FS_CD_ONE_LAUNCH, (turn, graph)
            return r

        a, b, e = run(False), run(True), run(True)
        assert e["graph_build_ms"] == 0.0  # a replay
        for r in (b, e):
            assert np.array_equal(a["U"], r["U"]) and np.array_equal(a["V"], r["V"]), turn
    f._model.close()
