"""Results into ordinary and into pinned host memory: the same values, at sizes of
one chunk of the copy, several chunks, and more chunks than slots; and into pinned
memory without a second pass over it on the host (a copy through the library's own
pinned chunks takes 1.4 times the direct one at 20 and 60 MB)."""
import ctypes as C
import time

import numpy as np
import pytest

from flexshell import _lib, fe, femm as FM
from flexshell.material import MatDeforElastIso

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


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
    best = {}
    pinned = torch.zeros(K.nnz, dtype=torch.float64, pin_memory=True).numpy()
    assert torch.from_numpy(pinned).is_pinned()
    # a range that begins inside the pinned block
    offset = torch.zeros(K.nnz + 5, dtype=torch.float64, pin_memory=True).numpy()[5:]
    for name, out in (("pinned", pinned), ("offset", offset), ("touched", np.zeros(K.nnz))):
        best[name] = np.inf
        for _ in range(6):
            out[:] = 0.0
            t = time.perf_counter()
            ctx.check(ctx.lib.fs_model_stiffness(f._model.h, C.byref(par), _lib.FS_BLOCK_FF, _lib.ptr(out)), "stiffness")
            best[name] = min(best[name], time.perf_counter() - t)
        assert np.array_equal(out, K.data), name
    if K.nnz * 8 > 40e6:
        assert best["pinned"] < 0.9 * best["touched"], best
    f._model.close()
