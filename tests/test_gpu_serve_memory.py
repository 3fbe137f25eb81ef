"""The footprint by which a request is admitted against the device memory it takes:
all buffers that its context has allocated for it (a fresh context keeps them as spare
buffers, so none are given back before the measurement)."""
import numpy as np
import pytest

from flexshell import _lib, fe, serve as S
from flexshell.material import MatDeforElastIso

pytestmark = pytest.mark.gpu

KINDS = [(S.ASSEMBLY, 0), (S.MODAL, 0)] + [(S.EXPLICIT, p) for p in (_lib.FS_PREC_FP64, _lib.FS_PREC_MIXED,
                                                                     _lib.FS_PREC_MIXED_F32)]


@pytest.mark.parametrize("nen, nx, ny", [(3, 100, 100), (4, 141, 141), (3, 360, 350), (4, 360, 350)])
def test_footprint_covers_the_request(ctx, nen, nx, ny):
    print(f"[gpu] footprints {nen} {nx}x{ny}", flush=True)
    xy, conn = (fe.T3block if nen == 3 else fe.Q4block)(0.1 * nx, 0.1 * ny, nx, ny)
    xyz = fe.xyz3(xy)
    d = fe.DofField(len(xyz))
    d.setebc(np.nonzero(xy[:, 0] < 1e-9)[0], [1, 2, 3])
    d.numberdofs()
    m = dict(xyz=xyz, conn=conn, dchi=d, material=MatDeforElastIso(70e9, 0.33, 2700.0), t=0.02)
    S.execute(S.Request(0, S.EXPLICIT, m, steps=100, precision=_lib.FS_PREC_MIXED), ctx)  # kernels' own memory
    for kind, precision in KINDS:
        c = S.request_context(ctx.device)
        before = S.device_memory(ctx.device)[0]
        r = S.Request(0, kind, m, steps=100, precision=precision)
        S.execute(r, c)
        used = before - S.device_memory(ctx.device)[0]
        c.close()
        assert 0 < used <= r.footprint, (kind, precision, used, r.footprint)
        assert r.footprint <= 2.5 * used, (kind, precision, used, r.footprint)
