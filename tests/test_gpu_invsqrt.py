"""S^-1/2 of lowdin at the edges of its tiles and K groups, against the
eigendecomposition.  The input is an orthonormal set plus a perturbation of norm
below 1/4, so that S is well conditioned; the errors are K u of the overlap, a few
n u of the last products of the iteration and n u of C Z, K = 2 ngw, on rows of C
of norm about 1: (2 K + 40 n) u, u = 2^-53, covers them and the reference's own."""
import numpy as np
import pytest

from cpmd_amd import ops
from cpmd_amd import system as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 127, 128, 129, 200, 257, 385])
def test_lowdin_edges(gpu, n):
    sysm = S.make_system(9.0, 8, 30.0, nstate=1)
    ngw = sysm.gset.ngw
    rng = np.random.default_rng(n)
    # real embedding of the half sphere: <a|b> = a0 b0 + 2 Re sum conj(a) b
    x = np.linalg.qr(rng.standard_normal((2 * ngw - 1, n)))[0]
    x += 0.1 * rng.standard_normal(x.shape) / np.sqrt(x.shape[0])
    w, q = np.linalg.eigh(x.T @ x)
    assert w[0] > 0.5 and w[-1] < 1.6
    ref = x @ (q / np.sqrt(w)) @ q.T

    def pack(v):
        c = np.zeros((ngw, n), np.complex128, order="F")
        c[0] = v[0]
        c[1:] = (v[1::2] + 1j * v[2::2]) / np.sqrt(2)
        return c

    out = ops.Context(sysm.cell, sysm.gset).lowdin(pack(x))
    assert np.abs(out - pack(ref)).max() < (4 * ngw + 40 * n) * 2.0 ** -53


def test_lowdin_nan(gpu):
    """A NaN among the coefficients is refused, not iterated on."""
    sysm = S.make_system(9.0, 8, 30.0, nstate=1)
    c = np.asfortranarray(np.eye(sysm.gset.ngw, 40, k=-1, dtype=np.complex128))
    c[5, 3] = np.nan
    with pytest.raises(Exception, match="non-finite"):
        ops.Context(sysm.cell, sysm.gset).lowdin(c)
