"""Orthonormalisation (lowdin, rgs) of sets whose overlap is far from the unit matrix (start
orbitals, large steps): S = P diag(w) P^T with a geometric spectrum from 1 / cond
to 1, C = Q diag(sqrt w) P^T with orthonormal Q."""
import numpy as np
import pytest

from cpmd_amd import ops
from cpmd_amd import system as S

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


@pytest.fixture(scope="module")
def sysm():
    return S.make_system(12.0, 8, 40.0, nstate=1)


def _set(sysm, n, cond, seed):
    """C packed to the half sphere (<a|b> = a0 b0 + 2 Re sum conj(a) b) and its real
    rows' polar factor Q P^T."""
    ngw = sysm.gset.ngw
    rng = np.random.default_rng(seed)
    q = np.linalg.qr(rng.standard_normal((2 * ngw - 1, n)))[0]
    p = np.linalg.qr(rng.standard_normal((n, n)))[0]
    w = np.geomspace(1.0 / cond, 1.0, n)
    return _pack((q * np.sqrt(w)) @ p.T), _pack(q @ p.T)


def _pack(x):
    c = np.zeros(((x.shape[0] + 1) // 2, x.shape[1]), np.complex128, order="F")
    c[0] = x[0]
    c[1:] = (x[1::2] + 1j * x[2::2]) / np.sqrt(2)
    return c


# K u of the overlap and a few n u of the last products, as for a well conditioned
# set; an error of that size in S moves S^-1/2 C by up to cond times it
def _tol(sysm, n, cond):
    return (4 * sysm.gset.ngw + 40 * n) * U * cond


@pytest.mark.parametrize("cond", [1e2, 1e3, 1e4, 1e6])
@pytest.mark.parametrize("n", [16, 67, 130, 257, 1025])
def test_lowdin(gpu, sysm, n, cond):
    """The coupled iteration holds only while its products are those of the factors
    in their order: formed as A^T B, or one triangle mirrored, it diverges from a
    condition of 1e2 or 1e3 on."""
    ctx = ops.Context(sysm.cell, sysm.gset)
    c, ref = _set(sysm, n, cond, n)
    d = ctx.upload(c)
    iters = ctx.lowdin_dev(d, n)
    assert iters <= 40
    assert np.abs(ctx.download(d, n) - ref).max() < _tol(sysm, n, cond)


@pytest.mark.parametrize("n", [2, 16, 17, 33, 50, 65, 130, 200])
def test_rgs(gpu, sysm, n):
    """C U^-1 is the Q of C = Q R with a positive diagonal; n at the edges of the
    16-row panels and 64-wide blocks of the factorisation."""
    ctx = ops.Context(sysm.cell, sysm.gset)
    c, _ = _set(sysm, n, 1e6, n)
    x = np.zeros((2 * sysm.gset.ngw - 1, n))
    x[0], x[1::2], x[2::2] = c[0].real, np.sqrt(2) * c[1:].real, np.sqrt(2) * c[1:].imag
    q, r = np.linalg.qr(x)
    g, smat = ctx.rgs(c)
    assert np.abs(g - _pack(q * np.sign(np.diag(r)))).max() < _tol(sysm, n, 1e6)
    assert not np.tril(smat, -1).any() and (np.diag(smat) > 0).all()
