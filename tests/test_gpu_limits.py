"""The FP64 projector and overlap products under a device memory limit that does
not hold what they take without one."""
import numpy as np
import pytest

from cpmd_amd import ops
from cpmd_amd import system as S

pytestmark = pytest.mark.gpu
N, NA, NHXS = 96, (30, 34), 4


def _ctx(sysm):
    rng = np.random.default_rng(6)
    ngw, nat = sysm.gset.ngw, sum(NA)
    ctx = ops.Context(sysm.cell, sysm.gset)
    lang = np.array([[0, 1], [1, 2], [1, 0], [2, 0]], np.int32, order="F")
    ctx.set_projectors(list(NA), NHXS, [4, 2], lang, rng.standard_normal((4, 4, 2)), rng.standard_normal((ngw, 4, 2)))
    ctx.set_eigr(np.asfortranarray(np.exp(2j * np.pi * rng.random((ngw, nat)))))
    gk = rng.standard_normal((3, ngw))
    gk[:, 0] = 0.0
    ctx.set_gk(gk)
    c = rng.standard_normal((ngw, N)) + 1j * rng.standard_normal((ngw, N))
    c[0] = c[0].real
    return ctx, ctx.upload(np.asfortranarray(c)), ctx.upload(np.asfortranarray(c[:, ::-1]))


# Two orders of a sum of K random products differ by at most 2 K u sum |a| |b|, and
# that sum is below sqrt K times the largest of the results
def _tol(sysm):
    k = 2 * sysm.gset.ngw
    return 2 * k * 2.0 ** -53 * np.sqrt(k)


# fnl and dfnl, and beside them as many bytes as a product per species and projector
# takes (34 columns, the K = 7250 rows split 14 times), or only the sums of 10 columns
# without a split
@pytest.mark.parametrize("beside", [8 * N * 34 * 14, 8 * N * 10])
def test_projectors(gpu, beside):
    sysm = S.make_system(12.0, 8, 40.0, nstate=1)
    f = np.full(N, 2.0)
    got = []
    for limited in (False, True):
        ctx, d, d2 = _ctx(sysm)
        if limited:
            ops.set_mem_limit(ops.mem_stats()[0] + 8 * N * sum(NA) * NHXS * 4 + 4096 + beside)
        try:
            fnl, dfnl = ctx.rnlsm_dev(d, N, tfor=True, want_fnl=True, want_dfnl=True)
            if beside > 8 * N * 34:   # fnonloc's factors of one projector, behind the sums
                ops.set_mem_limit(limited and ops.mem_stats()[0] + 8 * N * 34 + 4096)
                ctx.fnonloc_dev(d2, f, N)
            ops.set_mem_limit(0)   # the download has a buffer of its own
            got.append((fnl, dfnl, ctx.download(d2, N)))
        finally:
            ops.set_mem_limit(0)
        ctx.close()
    for a, b in zip(*got):
        assert np.abs(a - b).max() <= _tol(sysm) * np.abs(a).max()


def test_overlap(gpu):
    sysm = S.make_system(12.0, 8, 40.0, nstate=1)
    got = []
    for limited in (False, True):
        ctx, d, d2 = _ctx(sysm)
        if limited:
            ops.set_mem_limit(ops.mem_stats()[0] + 3 * 8 * N * N)
        try:
            got.append(ctx.ovlap_dev(d, d2, N))
        finally:
            ops.set_mem_limit(0)
        ctx.close()
    assert np.abs(got[0] - got[1]).max() <= _tol(sysm) * np.abs(got[0]).max()
