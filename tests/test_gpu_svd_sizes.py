"""The bond SVD at the sizes where its kernels change shape, against LAPACK.

One two-site update of a random (non-canonical) pair of sites with graded Schmidt values and no
truncation: theta = U S V^H is then the gated product itself, so lambda must be its normalised
singular values and lambda_l Gamma_l lambda Gamma_r lambda_r the normalised product.

Sizes: both sides below 64 (the whole solve in one launch) with one pair of column blocks (up to
32 columns) and two, at the edges of both and of a 16-column block; a side of 64 and more
(pivoted QR, then the sweep-by-sweep solve) at the row counts where the QR panel takes more waves
or rows per thread (128, 256, 512) and one beyond each, with ranks from one partial block up.

Tolerances, fixed before the first run: a backward stable SVD of an m x n matrix has singular
values within a few eps ||theta||; the Jacobi's stopping bound adds 1e-13 per column pair, so
1e-12 on lambda and 1e-11 on the product (norm 1) hold with room for m = 516.
"""
import numpy as np
import pytest

from tebd_amd import Context

pytestmark = pytest.mark.gpu

SMALL = [(2, 1, 1, 1), (2, 4, 3, 8), (2, 8, 8, 8), (2, 8, 9, 9), (2, 16, 16, 16), (2, 16, 20, 17), (2, 31, 24, 17),
         (2, 24, 24, 24), (3, 5, 7, 21), (3, 21, 21, 21), (2, 31, 31, 31)]
LARGE = [(2, 32, 32, 32), (2, 1, 2, 64), (3, 43, 11, 3), (2, 64, 33, 9), (3, 43, 40, 20), (4, 64, 30, 16), (6, 43, 20, 8),
         (8, 64, 20, 6), (6, 86, 30, 12), (5, 13, 60, 45)]


@pytest.mark.parametrize("d,chil,chic,chir", SMALL + LARGE)
def test_svd_of_every_kernel_shape(d, chil, chic, chir):
    rng = np.random.default_rng([d, chil, chic, chir])
    m, n = d * chil, d * chir
    chi = max(chil, chic, chir, min(m, n))

    def cplx(*shape):
        return rng.normal(size=shape) + 1j * rng.normal(size=shape)

    def lam(k):
        v = np.sort(10.0 ** rng.uniform(-5, 0, k))[::-1]
        return v / np.linalg.norm(v)

    ll, lc, lr = lam(chil), lam(chic), lam(chir)
    gl, gr = cplx(chil, d, chic), cplx(chic, d, chir)          # a, i, b
    op = np.linalg.qr(cplx(d * d, d * d))[0]
    gam = np.zeros((2, chi, d, chi), np.complex128)            # site, b, i, a
    gam[0, :chic, :, :chil] = gl.transpose(2, 1, 0)
    gam[1, :chir, :, :chic] = gr.transpose(2, 1, 0)
    lams = np.zeros((3, chi))
    for row, v in zip(lams, (ll, lc, lr)):
        row[:v.size] = v
    theta = np.tensordot(ll[:, None, None] * gl * lc, gr * lr, (2, 0))                       # a k l b
    theta = np.tensordot(op.reshape(d, d, d, d), theta, ((2, 3), (1, 2))).transpose(2, 0, 1, 3)  # a i j b
    theta /= np.linalg.norm(theta)
    s = np.linalg.svd(theta.reshape(chil * d, d * chir), compute_uv=False)

    print(f"[gpu] svd {m} x {n}, middle {chic}", flush=True)
    with Context(2, d, chi, mode="fp64") as ctx:
        ctx.upload(gam, lams)
        trunc = ctx.two_site_op(1, op)
        k = int(ctx.bond_dims()[1])
        g, l = ctx.download(chi)
    assert trunc < 1e-12
    ref = np.zeros(chi)
    ref[:s.size] = s
    assert np.max(np.abs(l[1] - ref)) < 1e-12
    left = ll[:, None, None] * g[0, :k, :, :chil].transpose(2, 1, 0)
    right = g[1, :chir, :, :k].transpose(2, 1, 0) * lr
    assert np.linalg.norm(np.tensordot(left * l[1, :k], right, (2, 0)) - theta) < 1e-11
