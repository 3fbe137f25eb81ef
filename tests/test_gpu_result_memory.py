"""Results into ordinary and into pinned host memory: the same values, at sizes of
one chunk of the copy, several chunks, and more chunks than slots."""
import ctypes as C

import numpy as np
import pytest

import test_gpu_no_memory as NM
from flexshell import _lib, fe, femm as FM
from flexshell.material import MatDeforElastIso

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx, ny", [(9, 7), (60, 41), (160, 150)])
def test_values_into_pinned_memory(ctx, nx, ny):
    print(f"[gpu] result memory {nx}x{ny}", flush=True)
    xy, conn = fe.Q4block(0.1 * nx, 0.1 * ny, nx, ny)
    xyz = fe.xyz3(xy)
    d = fe.DofField(len(xyz)).numberdofs()
    f = FM.make(conn, MatDeforElastIso(70e9, 0.33, 2700.0), thickness=0.02, ctx=ctx)
    f.associategeometry(xyz)
    K = f.stiffness(FM.SysmatAssemblerFFBlock(d.nfreedofs), xyz, None, None, d)
    par = f._shell_params()
    p, hip = C.c_void_p(), C.CDLL("libamdhip64.so.7")  # the runtime that the library is linked with
    assert hip.hipHostMalloc(C.byref(p), C.c_size_t(8 * K.nnz + 40), C.c_uint(0)) == 0
    block = np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_double)), (K.nnz + 5,))
    pinned, offset = block[:-5], block[5:]  # the second begins inside the block
    for name, out in (("pinned", pinned), ("offset", offset), ("touched", np.zeros(K.nnz))):
        for _ in range(3):
            out[:] = 0.0
            ctx.check(ctx.lib.fs_model_stiffness(f._model.h, C.byref(par), _lib.FS_BLOCK_FF, _lib.ptr(out)), "stiffness")
            assert np.array_equal(out, K.data), name
    f._model.close()
    del block, pinned, offset, out
    assert hip.hipHostFree(p) == 0


def test_pinned_memory_takes_the_copy_itself(tmp_path):
    """A second pass over the bytes on the host would need the library's own pinned
    chunks for them; in a process whose hipHostMalloc is counted it makes none."""
    print("[gpu] result memory, direct copy", flush=True)
    NM._run(tmp_path, """
        shim.pinned.restype = C.c_size_t
        xy, conn = fe.Q4block(10.0, 9.0, 100, 90)
        xyz = fe.xyz3(xy)
        d = fe.DofField(len(xyz)).numberdofs()
        f = FM.make(conn, MatDeforElastIso(70e9, 0.33, 2700.0), thickness=0.02, ctx=ctx)
        f.associategeometry(xyz)
        f.stiffness(FM.SysmatAssemblerHIP(_lib.FS_BLOCK_FF), xyz, None, None, d)
        nnz = C.c_int64()
        ctx.check(ctx.lib.fs_model_pattern(f._model.h, _lib.FS_BLOCK_FF, None, C.byref(nnz)), "pattern")
        nnz = nnz.value
        assert 8 * nnz > 20e6
        hip, p = C.CDLL("libamdhip64.so.7"), C.c_void_p()
        assert hip.hipHostMalloc(C.byref(p), C.c_size_t(8 * nnz), C.c_uint(0)) == 0
        par, before = f._shell_params(), shim.pinned()
        out = np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_double)), (nnz,))
        call = lambda a: ctx.check(ctx.lib.fs_model_stiffness(f._model.h, C.byref(par), _lib.FS_BLOCK_FF, _lib.ptr(a)), "K")
        call(out)
        assert shim.pinned() == before
        touched = np.zeros(nnz)
        call(touched)
        assert shim.pinned() > before and np.array_equal(out, touched)
        f._model.close()
        print("done")
    """)
