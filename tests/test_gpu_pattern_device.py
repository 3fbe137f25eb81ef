"""Patterns made on the device and results copied out in pinned chunks, at the
sizes where the copy changes its form: one chunk, several, more chunks than
slots, and more columns than one window.  The columns are compared with the
structural union built with scipy (equal), the values with their transpose
(bitwise: both triangles come from one sum)."""
import numpy as np
import pytest
import scipy.sparse as sp

import test_gpu_cd_forms as CF
from flexshell import _lib, femm as FM
from flexshell.material import MatDeforElastIso

pytestmark = pytest.mark.gpu


def _reference(conn, dofnums, nrows):
    """Union of the element dof pairs below nrows (counts in 32 bits: a hub may
    have a multiple of 256 elements)."""
    E, nen = conn.shape
    inc = sp.csr_matrix((np.ones(E * nen, dtype=np.int32), (np.repeat(np.arange(E), nen), conn.ravel())),
                        shape=(E, dofnums.shape[0]))
    adj = (inc.T @ inc).tocoo()
    r = np.repeat(dofnums[adj.row], 6, axis=1)
    c = np.tile(dofnums[adj.col], (1, 6))
    keep = (r < nrows) & (c < nrows)
    pat = sp.csr_matrix((np.ones(int(keep.sum()), dtype=np.int8), (r[keep], c[keep])), shape=(nrows, nrows))
    pat.sort_indices()
    return pat


class _Dofs:
    def __init__(self, dofnums, nfree):
        self.dofnums, self.nfreedofs, self.nalldofs = dofnums, nfree, dofnums.size


def _plate(nen, nx, ny, seed):
    """Flat plate, its nodes shuffled, one edge simply supported: free dofs
    numbered first in node order, then the fixed ones."""
    X, Y = np.meshgrid(np.linspace(0, 2.0, nx + 1), np.linspace(0, 1.0, ny + 1), indexing="ij")
    N = X.size
    new = np.random.default_rng(seed).permutation(N)
    xyz = np.zeros((N, 3))
    xyz[new, 0], xyz[new, 1] = X.ravel(), Y.ravel()
    i, j = np.meshgrid(np.arange(nx), np.arange(ny), indexing="ij")
    a = (i * (ny + 1) + j).ravel()
    b, c, d = a + ny + 1, a + ny + 2, a + 1
    conn = np.stack([a, b, c, d], 1) if nen == 4 else np.vstack([np.stack([a, b, c], 1), np.stack([a, c, d], 1)])
    fixed = np.zeros((N, 6), dtype=bool)
    fixed[new[: ny + 1], :3] = True
    dofs = np.empty((N, 6), dtype=np.int64)
    nf = int((~fixed).sum())
    dofs[~fixed] = np.arange(nf)
    dofs[fixed] = np.arange(nf, 6 * N)
    return xyz, new[conn], _Dofs(dofs, nf)


# entries of the block: 30 thousand to 10 million (0.25 to 80 MB of columns)
@pytest.mark.parametrize("nen, nx, ny, ff", [(4, 9, 9, False), (3, 30, 20, True), (4, 60, 41, False),
                                             (3, 150, 120, True), (3, 210, 190, False)])
def test_pattern_and_values_by_size(ctx, nen, nx, ny, ff):
    print(f"[gpu] pattern by size {nen} {nx}x{ny} ff={ff}", flush=True)
    xyz, conn, d = _plate(nen, nx, ny, nx)
    cls = FM.FEMMShellT3FF if nen == 3 else FM.FEMMShellQ4RS
    f = cls(conn, MatDeforElastIso(210e9, 0.3, 7850.0), thickness=0.01, ctx=ctx)
    f.associategeometry(xyz)
    nf, na = d.nfreedofs, d.nalldofs
    asm = FM.SysmatAssemblerFFBlock(nf) if ff else FM.SysmatAssemblerSparseCSRSymm()
    K = f.stiffness(asm, xyz, None, None, d)
    P = _reference(conn, d.dofnums, nf if ff else na)
    assert K.shape == P.shape
    assert np.array_equal(K.indptr, P.indptr) and np.array_equal(K.indices, P.indices)
    KT = K.T.tocsr()
    KT.sort_indices()
    assert np.array_equal(KT.data, K.data)
    assert np.all(K.diagonal() > 0.0)
    nr, rp, cv = f._model.pattern(_lib.FS_BLOCK_FF)
    Pf = _reference(conn, d.dofnums, nf)
    assert np.array_equal(rp, Pf.indptr) and np.array_equal(cv, Pf.indices)


def _fan_q4(m):
    """m quadrilaterals around node 0, the outer nodes fixed."""
    ang = np.pi * np.arange(2 * m) / m
    r = np.where(np.arange(2 * m) % 2 == 0, 0.6, 1.0)
    xyz = np.vstack([[0.0, 0.0, 0.0], np.column_stack([r * np.cos(ang), r * np.sin(ang), 0.02 * np.cos(3 * ang)])])
    i = np.arange(m)
    conn = np.stack([0 * i, 1 + 2 * i, 2 + 2 * i, 1 + (2 * i + 2) % (2 * m)], 1)
    N = len(xyz)
    fixed = np.zeros((N, 6), dtype=bool)
    fixed[2::2] = True
    dofs = np.empty((N, 6), dtype=np.int64)
    nf = int((~fixed).sum())
    dofs[~fixed], dofs[fixed] = np.arange(nf), np.arange(nf, 6 * N)
    return 4, xyz, conn, _Dofs(dofs, nf)


# A hub's elements, where the planning changes its form: 15 | 16 triangles and 10 |
# 11 quadrilaterals (neighbour lists by the kernel or the host), 64 | 65 elements (two
# ways to intersect their lists), 255 | 256 spokes (the hub's list ordered by the
# kernel or the host), and far past all of these.
@pytest.mark.parametrize("nen, spokes", [(3, 15), (3, 16), (4, 10), (4, 11), (3, 64), (3, 65), (3, 255), (3, 256),
                                         (3, 700)])
@pytest.mark.parametrize("mode", [0, 1])
def test_hub(ctx, nen, spokes, mode):
    print(f"[gpu] hub of {spokes} nen {nen} mode {mode}", flush=True)
    nen, xyz, conn, d = CF._fan_t3(spokes) if nen == 3 else _fan_q4(spokes)
    cls = FM.FEMMShellT3FF if nen == 3 else FM.FEMMShellQ4RS
    ctx.set_assembly(mode)
    try:
        f = cls(conn, MatDeforElastIso(210e9, 0.3, 7850.0), thickness=0.01, ctx=ctx)
        f.associategeometry(xyz)
        Ke = f.element_matrices(xyz, d)
        for asm, n in ((FM.SysmatAssemblerFFBlock(d.nfreedofs), d.nfreedofs),
                       (FM.SysmatAssemblerSparseCSRSymm(), d.nalldofs)):
            K = f.stiffness(asm, xyz, None, None, d)
            P = _reference(conn, d.dofnums, n)
            assert np.array_equal(K.indptr, P.indptr) and np.array_equal(K.indices, P.indices)
            q = d.dofnums[conn].reshape(len(conn), 6 * nen)
            r, c = np.repeat(q, 6 * nen, axis=1).ravel(), np.tile(q, (1, 6 * nen)).ravel()
            keep = (r < n) & (c < n)
            S, A = (sp.coo_matrix((v.ravel()[keep], (r[keep], c[keep])), shape=(n, n)).toarray()
                    for v in (Ke, np.abs(Ke)))
            # each sum of at most `spokes` terms is within spokes * eps of the sum of magnitudes
            assert np.all(np.abs(K.toarray() - S) <= 2 * spokes * np.finfo(float).eps * A)
    finally:
        ctx.set_assembly(1)
