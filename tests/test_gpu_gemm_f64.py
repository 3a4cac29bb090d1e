"""The FP64 contractions at the edges of their tiles, entry by entry against
the sums in extended precision.  A K-term sum of products in FP64, in whatever
order, is off by at most K u sum |a| |b| to first order (u = 2^-53); twice
that covers the higher orders and the final scaling."""
import numpy as np
import pytest

from cpmd_amd import ops
from cpmd_amd import system as S

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


@pytest.fixture(scope="module")
def sysm():
    s = S.make_system(9.0, 8, 30.0, nstate=1)
    assert (2 * s.gset.ngw) % 16 != 0          # the last K slice is cut
    return s


def _wfn(sysm, n, seed):
    rng = np.random.default_rng(seed)
    ngw = sysm.gset.ngw
    c = np.asfortranarray(rng.standard_normal((ngw, n)) + 1j * rng.standard_normal((ngw, n)))
    c[0] = c[0].real
    return c


def _rows(c):
    return np.ascontiguousarray(c.T).view(np.float64)        # (n, 2 ngw)


@pytest.mark.parametrize("n", [1, 2, 31, 33, 64, 65, 96, 97, 129, 130, 161])
def test_ovlap_edges(gpu, sysm, n):
    ctx = ops.Context(sysm.cell, sysm.gset)
    a, b = _wfn(sysm, n, 1), _wfn(sysm, n, 2)
    for x, y in ((a, a), (a, b)):
        rx, ry = _rows(x).astype(np.longdouble), _rows(y).astype(np.longdouble)
        ref = 2 * (rx @ ry.T) - np.outer(rx[:, 0], ry[:, 0])
        mag = (2 * (np.abs(rx) @ np.abs(ry).T)).astype(np.float64)
        s = ctx.ovlap(x, x if y is x else y)
        assert np.all(np.abs(s - ref) <= 2 * (rx.shape[1] + 8) * U * mag)
        if y is x:
            assert np.array_equal(s, s.T)


@pytest.mark.parametrize("n", [2, 15, 33, 64, 97, 130, 161])
def test_rotate_edges(gpu, n):
    sysm = S.make_system(12.0, 8, 40.0, nstate=1)            # enough rows for the tall kernel
    ctx = ops.Context(sysm.cell, sysm.gset)
    a, b = _wfn(sysm, n, 3), _wfn(sysm, n, 4)
    g = np.random.default_rng(5).standard_normal((n, n))
    for beta in (0.0, -0.75):
        out = ctx.rotate(1.5, a, beta, b, g)
        lg = g.astype(np.longdouble)
        for part in ("real", "imag"):
            la, lb = getattr(a, part).astype(np.longdouble), getattr(b, part).astype(np.longdouble)
            ref = 1.5 * (la @ lg) + beta * lb
            mag = (1.5 * (np.abs(la) @ np.abs(lg)) + abs(beta) * np.abs(lb)).astype(np.float64)
            assert np.all(np.abs(getattr(out, part) - ref) <= 2 * (n + 8) * U * mag)


@pytest.mark.parametrize("n", [250, 256])
def test_rotate_wide_tiles(gpu, n):
    """Enough rows for the 64-wide tiles (2048 of them), odd rows left over."""
    sysm = S.make_system(30.0, 1, 30.0, nstate=1)
    assert (2 * sysm.gset.ngw + 127) // 128 * 4 >= 2048
    a, b = _wfn(sysm, n, 3), _wfn(sysm, n, 4)
    g = np.random.default_rng(5).standard_normal((n, n))
    out = ops.Context(sysm.cell, sysm.gset).rotate(1.5, a, -0.75, b, g)
    rows = np.r_[0:sysm.gset.ngw:97, sysm.gset.ngw - 70:sysm.gset.ngw]
    lg = g.astype(np.longdouble)
    for part in ("real", "imag"):
        la, lb = getattr(a, part)[rows].astype(np.longdouble), getattr(b, part)[rows].astype(np.longdouble)
        ref = 1.5 * (la @ lg) - 0.75 * lb
        mag = (1.5 * (np.abs(la) @ np.abs(lg)) + 0.75 * np.abs(lb)).astype(np.float64)
        assert np.all(np.abs(getattr(out, part)[rows] - ref) <= 2 * (n + 8) * U * mag)


@pytest.mark.parametrize("na,n", [((1, 0), 1), ((3, 5), 17), ((0, 7), 64), ((21, 44), 33)])
def test_stacked_projectors(gpu, sysm, na, n):
    """fnl, dfnl and fnonloc over several species and projectors (l = 0 .. 3, a
    species with fewer projectors than nhxs, a species without atoms)."""
    rng = np.random.default_rng(6)
    ngw, nat = sysm.gset.ngw, sum(na)
    ngh = [4, 2]
    lang = np.array([[0, 1], [1, 2], [2, 0], [3, 0]], np.int32, order="F")
    tw = np.asfortranarray(rng.standard_normal((ngw, 4, 2)))
    h = np.asfortranarray(rng.standard_normal((4, 4, 2)))
    eigr = np.asfortranarray(np.exp(2j * np.pi * rng.random((ngw, nat))))
    gk = rng.standard_normal((3, ngw))
    gk[:, 0] = 0.0
    c, f = _wfn(sysm, n, 7), np.where(np.arange(n) % 5 == 3, 0.0, 2.0)
    ctx = ops.Context(sysm.cell, sysm.gset)
    ctx.set_projectors(list(na), 4, ngh, lang, h, tw)
    ctx.set_eigr(eigr)
    ctx.set_gk(gk)
    d = ctx.upload(c)
    fnl, dfnl = ctx.rnlsm_dev(d, n, tfor=True, want_fnl=True, want_dfnl=True)
    assert np.array_equal(fnl, ctx.rnlsm1_dev(d, n, want_fnl=True))
    assert np.array_equal(dfnl, ctx.rnlsm2_dev(d, n, want_dfnl=True))
    K, tpiba, ld = 2 * ngw, sysm.cell.tpiba, np.longdouble
    rc = _rows(c).astype(ld)
    add = np.zeros((ngw, n), np.clongdouble)
    mag_add = np.zeros((ngw, n))
    occ = np.where(f < 1e-5, 1.0, f)
    isa = 0
    for s in range(2):
        for ia in range(na[s]):
            for iv in range(4):
                if iv >= ngh[s]:
                    assert not fnl[isa, iv].any() and not dfnl[isa, iv].any()
                    continue
                beta = (-1j) ** int(lang[iv, s]) * tw[:, iv, s] * eigr[:, isa]
                for k in range(-1, 3):
                    b = beta.copy() if k < 0 else -1j * gk[k] * beta
                    b[0] *= 0.5
                    rb = b.view(np.float64).astype(ld)
                    ref = 2 * (rc @ rb) * (1.0 if k < 0 else tpiba)
                    mag = (2 * (np.abs(rc) @ np.abs(rb)) * (1.0 if k < 0 else tpiba)).astype(np.float64)
                    got = fnl[isa, iv] if k < 0 else dfnl[isa, iv, k]
                    assert np.all(np.abs(got - ref) <= 2 * (K + 8) * U * mag)
                dd = h[iv, :ngh[s], s] @ fnl[isa, :ngh[s]]
                mdd = np.abs(h[iv, :ngh[s], s]) @ np.abs(fnl[isa, :ngh[s]])
                add += -np.outer(beta, occ * dd)
                mag_add += np.outer(np.abs(beta), occ * mdd)
            isa += 1
    c2 = _wfn(sysm, n, 8)
    out = ctx.fnonloc(c2, f, fnl)
    terms = max(1, nat * 4)
    assert np.all(np.abs(out - (c2 + add)) <= 4 * (terms + 16) * U * (np.abs(c2) + mag_add))
