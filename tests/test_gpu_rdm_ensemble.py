"""All-pairs density matrices of an ensemble with more sites than a grid's second dimension is
specified to hold.

8200 chains of 8 spins: 65600 environments, while HIP gives 65536 as the most workgroups of a launch's
second and third dimensions.  On product states every matrix is the product of the two sites' own,
which is exact: 1e-13.
"""
import numpy as np
import pytest

from tebd_amd import Ensemble, models as M

pytestmark = pytest.mark.gpu


def test_more_sites_than_one_launch_holds():
    n, Lc, d, chi = 8200, 8, 2, 2
    rng = np.random.default_rng(n)
    c = rng.normal(size=(n, Lc, d)) + 1j * rng.normal(size=(n, Lc, d))
    c /= np.linalg.norm(c, axis=2, keepdims=True)
    gam, lam = M.product_state(c.reshape(n * Lc, d), 1)
    print(f"[gpu] density matrices of {n} chains", flush=True)
    with Ensemble(n, Lc, d, chi, mode="batched") as ens:
        ens.upload_chains(gam.reshape(n, Lc, 1, d, 1), np.ones((n, Lc + 1, 1)))
        rho2, rho1 = ens.two_point_rdms()
    site = np.einsum("rsi,rsj->rsij", c, c.conj())
    assert np.max(np.abs(rho1.reshape(n, Lc, d, d) - site)) < 1e-13
    for l1 in range(Lc):
        for l2 in range(l1 + 1, Lc):
            ref = np.einsum("rij,rkl->rikjl", site[:, l1], site[:, l2]).reshape(n, d * d, d * d)
            assert np.max(np.abs(rho2[:, l1, l2] - ref)) < 1e-13
