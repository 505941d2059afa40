"""Two-site expectation values at the edges of the kernel's tiles, against numpy.

<theta| O |theta> of random pairs of sites for every local dimension the kernel is built for, with
outer bond dimensions around one tile (16 states, 8 for d = 6 and 8) and a middle one around its
staging chunk (32).  A sum of at most d^2 chi^2 products, each from an FP64 dot product over the
middle bond: relative to ||theta|| ||O theta|| rounding stays below 1e-13 times a few; 1e-12.
"""
import numpy as np
import pytest

from tebd_amd import Context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [2, 3, 4, 5, 6, 8])
@pytest.mark.parametrize("dims", [(1, 1, 1, 1), (1, 7, 8, 9), (15, 31, 16, 33), (17, 32, 33, 1)])
def test_expval_tile_edges(d, dims):
    rng = np.random.default_rng([d, *dims])
    chi = max(dims)

    def cplx(*shape):
        return rng.normal(size=shape) + 1j * rng.normal(size=shape)

    G = [cplx(dims[s], d, dims[s + 1]) for s in range(3)]
    lam = [np.sort(rng.uniform(0.05, 1.0, k))[::-1] for k in dims]
    gam = np.zeros((3, chi, d, chi), np.complex128)
    lams = np.zeros((4, chi))
    for s in range(3):
        gam[s, :dims[s + 1], :, :dims[s]] = G[s].transpose(2, 1, 0)
    for row, v in zip(lams, lam):
        row[:v.size] = v
    ops = cplx(2, d * d, d * d)
    with Context(3, d, chi, mode="fp64") as ctx:
        ctx.upload(gam, lams)
        got = ctx.expval_two_site(ops)
    for b in range(2):
        th = np.tensordot(lam[b][:, None, None] * G[b] * lam[b + 1], G[b + 1] * lam[b + 2], (2, 0))
        oth = np.tensordot(ops[b].reshape(d, d, d, d), th, ((2, 3), (1, 2))).transpose(2, 0, 1, 3)
        assert abs(got[b] - np.vdot(th, oth)) < 1e-12 * np.linalg.norm(th) * np.linalg.norm(oth)
