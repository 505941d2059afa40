"""How orthogonal the singular vectors of small Schmidt values come out of a bond update.

One two-site operator (the identity) on a pair of sites whose theta = U diag(s) V^H has a generic
basis on both sides and s graded over 10 decades, all outer lambdas 1, nothing truncated: the new
Gammas are the singular vectors themselves.  The Jacobi stops when every pair of columns has
|w_p^H w_q| <= tol max|w| (|w_p| + |w_q|), so a pair of unit vectors is orthogonal to
2 tol s_max / min(s_p, s_q): two vectors of small values may be mixed by that angle, and the next
updates divide by those values.  (A pair also passes once |w_p^H w_q| <= 1e-13 |w_p| |w_q|, the looser
of the two where both values are within a factor of five of the largest: pairs with one below a tenth
of it are looked at.)

tol is 1e-14 where a pair visit is one pass of rotations (up to 512 rows), 1e-13 where it is whole
cyclic sweeps.  Bound, fixed before the first run: 2 tol, and a tenth of it for the rounding of the
vectors and of this test's products (1e-16 times a few).
"""
import numpy as np
import pytest

from tebd_amd import Context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,chil,chir", [(2, 32, 32), (2, 50, 53), (2, 113, 113), (3, 60, 75), (4, 64, 64), (4, 100, 97), (2, 256, 256),
                                         (2, 258, 258)])
@pytest.mark.parametrize("decades", [6, 10])
def test_small_vectors_are_orthogonal(d, chil, chir, decades):
    rng = np.random.default_rng([d, chil, chir, decades])
    m, n = d * chil, d * chir
    r = min(m, n)

    def basis(k):
        return np.linalg.qr(rng.normal(size=(k, r)) + 1j * rng.normal(size=(k, r)))[0]

    left, right = basis(m), basis(n).conj().T
    s = 10.0 ** -np.linspace(0, decades, r)
    s /= np.linalg.norm(s)
    chi = max(chil, chir, r)
    gam = np.zeros((2, chi, d, chi), np.complex128)                      # site, b, i, a
    gam[0, :r, :, :chil] = left.reshape(chil, d, r).transpose(2, 1, 0)
    gam[1, :chir, :, :r] = right.reshape(r, d, chir).transpose(2, 1, 0)
    lams = np.zeros((3, chi))
    lams[0, :chil] = lams[2, :chir] = 1.0
    lams[1, :r] = s
    print(f"[gpu] vectors of {m} x {n}, {decades} decades", flush=True)
    with Context(2, d, chi, mode="fp64") as ctx:
        ctx.upload(gam, lams)
        ctx.two_site_op(1, np.eye(d * d, dtype=np.complex128))
        g, l = ctx.download(chi)
    got = l[1, :r]
    assert np.max(np.abs(got - s)) < 1e-12
    tol = 1e-14 if r <= 512 else 1e-13
    small = np.minimum(got[:, None], got[None, :]) / got[0]
    for v in (g[0, :r, :, :chil].reshape(r, -1), g[1, :chir, :, :r].transpose(2, 1, 0).reshape(r, -1)):
        overlap = np.abs(v.conj() @ v.T - np.eye(r))
        assert np.max((overlap * small)[small < 0.1]) < 2.2 * tol
