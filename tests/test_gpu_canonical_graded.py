"""CanonicalForm of a bond whose site matrices are graded, against LAPACK.

Its SVDs run without QR preconditioning, so a Jacobi that is fast on preconditioned bonds can fail
to converge here.  Gamma1 = U diag(s) V^H with a generic basis and s from 1 down over the given
decades, Gamma2 with orthonormal rows, all outer lambdas 1: the canonical lambda is the normalised
spectrum of Gamma1 lambda Gamma2.  Sizes lie on both sides of the one-launch solve's bounds (32
columns, 64 rows) and where 40 sweeps get scarce (192 columns and more over 13 decades).

Tolerances, fixed before the first run: singular values of a backward stable SVD are off by a few
eps of the largest, the stopping bound adds 1e-13 per column pair: 1e-11 absolute.  The lambda
matrix is the product of two factors that carry s (the square roots of S1 and U1), each accurate to
1e-13 of the largest value; above 1e-2 of it that is 1e-9 relative with room.
"""
import numpy as np
import pytest

from tebd_amd import Context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,n,decades", [(2, 7, 3), (4, 31, 4), (4, 32, 13), (2, 33, 10), (8, 64, 13), (4, 65, 10), (4, 128, 13),
                                         (4, 192, 13), (4, 224, 13)])
def test_graded_bond(d, n, decades):
    rng = np.random.default_rng([n, d, decades, 0])
    q = -(-n // d)

    def cplx(*shape):
        return rng.normal(size=shape) + 1j * rng.normal(size=shape)

    U, V = np.linalg.qr(cplx(d * q, n))[0], np.linalg.qr(cplx(n, n))[0]
    left = (U * 10.0 ** -np.linspace(0, decades, n)) @ V.conj().T   # row i q + a
    right = np.linalg.qr(cplx(d * q, n))[0].conj().T                # column j q + b
    chi = max(n, q)
    gam = np.zeros((2, chi, d, chi), np.complex128)                 # site, b, i, a
    gam[0, :n, :, :q] = left.reshape(d, q, n).transpose(2, 0, 1)
    gam[1, :q, :, :n] = right.reshape(n, d, q).transpose(2, 1, 0)
    lam = np.zeros((3, chi))
    lam[0, :q] = lam[2, :q] = 1.0
    lam[1, :n] = 1.0 / np.sqrt(n)
    ref = np.linalg.svd(left @ right, compute_uv=False)[:n]
    ref /= np.linalg.norm(ref)
    print(f"[gpu] canonical form {d * q} x {n}, {decades} decades", flush=True)
    with Context(2, d, chi, mode="fp64") as ctx:
        ctx.upload(gam, lam)
        ctx.canonical_form(1)
        got = ctx.lambdas()[1][:n]
    got = got / np.linalg.norm(got)
    assert np.max(np.abs(got - ref)) < 1e-11
    big = ref > 1e-2 * ref[0]
    assert np.max(np.abs(got - ref)[big] / ref[big]) < 1e-9
