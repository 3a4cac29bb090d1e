"""rgs (blocked Cholesky, its inverse and the in-place product) at the edges of
the 64-wide blocks, and the order reported for a matrix that is not positive
definite."""
import numpy as np
import pytest
import scipy.linalg

from cpmd_amd import ops
from cpmd_amd._lib import McError
from cpmd_amd import system as S

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sysm():
    return S.make_system(12.0, 8, 40.0, nstate=1)


def _near_orthonormal(sysm, n, seed=1):
    rng = np.random.default_rng(seed)
    ngw = sysm.gset.ngw
    c = rng.standard_normal((ngw, n)) + 1j * rng.standard_normal((ngw, n))
    c[0] = c[0].real
    return np.asfortranarray(c / np.sqrt(4.0 * ngw))


@pytest.mark.parametrize("n", [1, 63, 64, 65, 127, 128, 129, 160, 161, 192, 257, 330])
def test_rgs_blocks(gpu, sysm, n):
    ctx = ops.Context(sysm.cell, sysm.gset)
    c = _near_orthonormal(sysm, n)
    s = S.dotp_gamma(c, c)
    u = scipy.linalg.cholesky(s)
    x = scipy.linalg.solve_triangular(u, np.eye(n))
    g, smat = ctx.rgs(c)
    # the condition number of S is below 10 (random vectors, ngw >> n): both sides
    # are within a few n u of the exact factor, times cond
    assert np.linalg.cond(s) < 10.0
    tol = 40 * (n + 16) * 2.0 ** -53 * np.abs(x).max()
    assert np.abs(smat - x).max() < tol
    assert not np.tril(smat, -1).any()
    ref = c @ x
    ref[0] = ref[0].real
    assert np.abs(g - ref).max() < tol * np.abs(c).max() * np.sqrt(n) * 4
    assert not g[0].imag.any()


@pytest.mark.parametrize("n,bad", [(5, 3), (100, 64), (130, 65), (200, 200), (200, 129)])
def test_not_positive_definite(gpu, sysm, n, bad):
    """A state of zeros: its pivot is exactly 0, the error names its order, and the
    coefficients are left as they were."""
    ctx = ops.Context(sysm.cell, sysm.gset)
    c = _near_orthonormal(sysm, n)
    c[:, bad - 1] = 0.0
    d = ctx.upload(c)
    with pytest.raises(McError) as e:
        ctx.rgs_dev(d, n)
    assert f"order {bad} " in str(e.value)
    assert np.array_equal(ctx.download(d, n), c)
