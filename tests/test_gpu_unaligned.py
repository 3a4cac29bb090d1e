"""Device wavefunctions that are only 8-byte aligned: the overlap and the projector
products take other kernels than for 16-byte aligned ones."""
import types

import numpy as np
import pytest

from cpmd_amd import ops
from cpmd_amd import system as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 17, 70])
def test_unaligned(gpu, n):
    sysm = S.make_system(9.0, 8, 30.0, nstate=1)
    rng = np.random.default_rng(n)
    ngw, na = sysm.gset.ngw, [3, 5]
    ctx = ops.Context(sysm.cell, sysm.gset)
    lang = np.array([[0, 1], [1, 2], [2, 3]], np.int32, order="F")
    ctx.set_projectors(na, 3, [3, 2], lang, rng.standard_normal((3, 3, 2)), rng.standard_normal((ngw, 3, 2)))
    ctx.set_eigr(np.asfortranarray(np.exp(2j * np.pi * rng.random((ngw, sum(na))))))
    gk = rng.standard_normal((3, ngw))
    gk[:, 0] = 0.0
    ctx.set_gk(gk)
    c = rng.standard_normal((ngw, n)) + 1j * rng.standard_normal((ngw, n))
    c[0] = c[0].real
    d = ctx.upload(np.asfortranarray(c))
    buf = ops.DeviceArray(d.nbytes + 8)
    buf.from_host(np.concatenate([[0.0], d.to_host(d.nbytes // 8)]))
    off = types.SimpleNamespace(ptr=type(buf.ptr)(buf.value + 8))
    # two orders of a sum of K products differ by at most 2 K u sum |a| |b|; for random
    # numbers that sum is below sqrt K times the largest result
    tol = 2 * (2 * ngw) * 2.0 ** -53 * np.sqrt(2 * ngw)
    for x, y in zip(ctx.rnlsm_dev(d, n, tfor=True, want_fnl=True, want_dfnl=True),
                    ctx.rnlsm_dev(off, n, tfor=True, want_fnl=True, want_dfnl=True)):
        assert np.abs(x - y).max() <= tol * np.abs(x).max()
    s = ctx.ovlap_dev(d, d, n)
    assert np.abs(ctx.ovlap_dev(off, off, n) - s).max() <= tol * np.abs(s).max()
