"""Calls that find no device memory.  A small library loaded before the HIP runtime
takes hipMalloc's place in a process of its own and refuses requests of given
sizes, as a full device does.  (It counts the bytes of hipHostMalloc too.)"""
import os
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = """
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
static size_t lo = 1, hi = 0;
static long refused = 0, first = 0;  /* the first requests of these sizes are granted */
void refuse(size_t a, size_t b, long skip) { lo = a; hi = b; refused = 0; first = skip; }
long refusals(void) { return refused; }
int hipMalloc(void **p, size_t n) {
    static int (*real)(void **, size_t);
    if (n >= lo && n <= hi && first-- <= 0) { ++refused; *p = 0; return 2; }  /* hipErrorOutOfMemory */
    if (!real) real = (int (*)(void **, size_t))dlsym(dlopen("libamdhip64.so.7", RTLD_NOW), "hipMalloc");
    return real(p, n);
}
static size_t host_bytes = 0;
size_t pinned(void) { return host_bytes; }
int hipHostMalloc(void **p, size_t n, unsigned flags) {
    static int (*real)(void **, size_t, unsigned);
    if (!real) real = (int (*)(void **, size_t, unsigned))dlsym(dlopen("libamdhip64.so.7", RTLD_NOW), "hipHostMalloc");
    host_bytes += n;
    return real(p, n, flags);
}
"""

HEAD = """
import ctypes as C, sys
shim = C.CDLL(sys.argv[1], C.RTLD_GLOBAL)
shim.refuse.argtypes = [C.c_size_t, C.c_size_t, C.c_long]
shim.refusals.restype = C.c_long
sys.path[:0] = [sys.argv[2], sys.argv[2] + "/finetoolsflexstructures.jl_amd"]
import numpy as np
from flexshell import _lib, explicit, fe, femm as FM
from flexshell.material import MatDeforElastIso
ctx = _lib.Context(0)
NONE, ALL = (1, 0), (0, 2 ** 63)
def refuse(r, skip=0): shim.refuse(*r, skip)
"""


def _run(tmp_path, script):
    c, so = tmp_path / "shim.c", tmp_path / "libshim.so"
    c.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", str(so), str(c), "-ldl"], check=True)
    r = subprocess.run([sys.executable, "-u", "-c", HEAD + textwrap.dedent(script), str(so), ROOT],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.strip().endswith("done"), r.stdout[-3000:]


@pytest.mark.gpu
def test_new_equation_numbers_need_no_memory(tmp_path):
    """The numbers of a model that has some go into the buffer that it has, also
    where the context keeps no more spare buffers (4 GiB of them here) and none is to
    be had."""
    print("[gpu] equation numbers without memory", flush=True)
    _run(tmp_path, """
        N = 2000000
        big = _lib.Model(ctx, 3, np.random.default_rng(0).random((N, 3)), np.array([[0, 1, 2]]))
        fixed = np.zeros((N, 6), dtype=np.uint8)
        dn, nf = big.number_dofs(fixed)
        ctx.set_assembly(0)
        models = []
        for _ in range(4):
            xy, conn = fe.Q4block(1.0, 1.0, 512, 512)
            xyz = fe.xyz3(xy)
            d = fe.DofField(len(xyz)).numberdofs()
            f = FM.make(conn, MatDeforElastIso(70e9, 0.33, 2700.0), thickness=0.02, ctx=ctx)
            f.associategeometry(xyz)
            f.stiffness(FM.SysmatAssemblerHIP(_lib.FS_BLOCK_FF), xyz, None, None, d)
            models.append(f)
        for f in models:
            f._model.close()
        # three nodes carry rows; the first pattern of the old numbers
        nr, rp, cv = big.pattern(_lib.FS_BLOCK_ALL)
        assert nr == 6 * N and len(cv) == 18 * 18
        refuse((90 * 10 ** 6, 2 ** 63))
        fixed[1] = 1
        dn2, nf2 = big.number_dofs(fixed)
        assert nf2 == nf - 6 and dn2[1].min() == nf2
        big.set_dofs(dn[::-1], 6 * N, nf)
        big.set_dofs(dn2, 6 * N, nf2)
        assert shim.refusals() == 0
        refuse(NONE)
        nr, rp, cv = big.pattern(_lib.FS_BLOCK_FF)
        assert nr == nf2 and len(cv) == 12 * 12
        big.close()
        print("done")
    """)


@pytest.mark.gpu
def test_loop_without_memory_for_its_patches(tmp_path):
    """The state of a loop on patches is padded to whole patches.  Where that finds no
    memory the row products take over (equal up to the order of addition), where
    only the words of the one-launch loop do not, the loop goes step by step (bitwise
    equal); where the row products find none either, the call fails, and the next
    one works."""
    print("[gpu] loop without memory", flush=True)
    _run(tmp_path, """
        for nx, ny, first in ((400, 300, _lib.FS_CD_PATCHES), (100, 90, _lib.FS_CD_ONE_LAUNCH)):
            xy, conn = fe.T3block(0.1 * nx, 0.1 * ny, nx, ny)
            xyz = fe.xyz3(xy)
            d = fe.DofField(len(xyz))
            d.setebc(np.nonzero(xy[:, 0] < 1e-9)[0], [1, 2, 3])
            d.numberdofs()
            n = d.nfreedofs
            nv = 252 * -(-len(xyz) // 42)
            rng = np.random.default_rng(0)
            U0, V0, F = rng.normal(0, 1e-6, n), rng.normal(0, 1e-3, n), rng.normal(0, 1.0, n)
            g, probes = np.cos(0.1 * np.arange(121)), np.array([0, n - 1, 77])

            def model():
                c = _lib.Context(0)  # no spare buffers
                f = FM.make(conn, MatDeforElastIso(70e9, 0.33, 2700.0), thickness=0.02, ctx=c)
                f.associategeometry(xyz)
                f.stiffness(FM.SysmatAssemblerHIP(_lib.FS_BLOCK_FF), xyz, None, None, d)
                f.mass(FM.SysmatAssemblerHIP(_lib.FS_BLOCK_FF), xyz, d)
                return f

            def loop(f, sizes, prec, graph=False, skip=0):
                refuse(sizes, skip)
                try:
                    r = explicit.run(f._model, 10.0, U0, V0, 2e-7, 120, F, g, probes, 10, prec, use_graph=graph)
                    return r, f._model.cd_form()
                finally:
                    refuse(NONE)

            for prec in (_lib.FS_PREC_FP64, _lib.FS_PREC_MIXED, _lib.FS_PREC_MIXED_F32):
                f = model()
                ref, form = loop(f, NONE, prec)
                assert form == first
                f._model.close()
                f = model()
                # the sizes of the state: of the patches' slots, not of the dofs, nodes or words
                state = (8 * nv, 8 * nv)
                try:
                    loop(f, (8 * min(n, nv), 8 * max(n, nv, 6 * len(xyz))), prec)
                    raise SystemExit("no error")
                except _lib.FlexShellError as e:
                    assert "out of memory" in str(e)
                f._model.close()
                f = model()
                for graph in (False, True, True):
                    # the plan's map of the slots has that size too, and is granted
                    r, form = loop(f, state, prec, graph, 1)
                    assert form == _lib.FS_CD_ROWS, form
                    for k in ("U", "V", "probes"):
                        assert np.linalg.norm(r[k] - ref[k]) <= 1e-11 * np.linalg.norm(ref[k]), k
                f._model.close()
                if first != _lib.FS_CD_ONE_LAUNCH:
                    continue
                f = model()
                for graph in (False, True):
                    r, form = loop(f, (32 * nv, 32 * nv), prec, graph)
                    assert form == _lib.FS_CD_PATCHES, form
                    assert all(np.array_equal(r[k], ref[k]) for k in ("U", "V", "probes"))
                r, form = loop(f, NONE, prec, True)
                assert form == first and np.array_equal(r["U"], ref["U"])
                f._model.close()
        print("done")
    """)
