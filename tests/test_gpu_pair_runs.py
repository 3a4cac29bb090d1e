"""vpsi with several state pairs per workgroup in its y and x passes: many pairs on a
small mesh.  Pairs are independent, so that the result is that of one pair per
call, bit for bit (which the other tests compare with the oracle)."""
import math

import numpy as np
import pytest

from cpmd_amd import ops
from cpmd_amd import system as S

pytestmark = pytest.mark.gpu


# FP64 with two LDS buffers (60) and with one (the others); FP32 four-step (54, 128) and
# stages of the plan, split nearly evenly (60) and not (80 = 16 x 5, 100 = 4 x 25)
@pytest.mark.parametrize("n", [54, 60, 80, 100, 128])
def test_vpsi_runs(gpu, n):
    ecut, nr = 4.0, (n, n, 16)
    edge = [(m - 0.6) * math.pi / math.sqrt(4.0 * ecut) for m in nr]
    cell = S.Cell(alat=edge[0], avec=np.diag(edge).astype(float), ecut=ecut, dual=4.0, nr=nr)
    gs = S.gvectors(cell, with_density=False)
    rng = np.random.default_rng(n)
    # the y pass aims at 65536 workgroups of (column, z tile, run of pairs), the x pass
    # at 1024 to 2047 of (z tile, row, run): beyond them a run is two pairs or more
    ncols = 2 * int(np.abs(gs.miller[:, 0]).max()) + 1
    pairs = 65536 // ncols + 30
    ctx = ops.Context(cell, gs)
    c = rng.standard_normal((gs.ngw, 2 * pairs)) + 1j * rng.standard_normal((gs.ngw, 2 * pairs))
    c[0] = c[0].real
    d, f = ctx.upload(np.asfortranarray(c)), rng.uniform(0.5, 2.0, 2 * pairs)
    v = ops.DeviceArray(8 * ctx.nnr1).from_host(rng.standard_normal(ctx.nnr1))
    for mode in ("fp64", "fp32"):
        ctx.set_precision(mode)
        got = []
        for batch in (pairs, 1):
            ctx.set_batch(batch, batch)
            out = ctx.upload(np.zeros_like(c, order="F"))
            ctx.vpsi_dev(d, out, f, v, 2 * pairs)
            got.append(ctx.download(out, 2 * pairs))
            out.free()
        assert np.array_equal(*got)
        assert np.abs(got[0]).max() > 0.0
