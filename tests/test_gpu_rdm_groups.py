"""All-pairs density matrices where the environments do not fit one group, and at the edges of
the contraction's lane and wave split.

A group holds the environments of as many right sites as fit its budget (4 GiB); 44 sites of
d = 8 with room for chi = 100 take two groups.  On a product state every pair's matrix is the
product of the two sites' own, |c><c|, which is exact; entries are sums of products of unit
vectors, so 1e-13 holds.

Entangled chains are compared with the CPU oracle's table at bond dimensions on both sides of
the contraction's splits (64 lanes over the right bond, four waves over the left one), for each
local dimension the kernel is built for and an ensemble of two chains.  Both sides contract the
same Gammas and lambdas (canonical to the Jacobi's 1e-13) over at most a few hundred terms of
norm at most one: 1e-11.
"""
import numpy as np
import pytest

from oracle.oracle import two_point_rdms
from tebd_amd import Context, Ensemble, models as M

pytestmark = pytest.mark.gpu


def random_product(rng, L, d):
    c = rng.normal(size=(L, d)) + 1j * rng.normal(size=(L, d))
    return c / np.linalg.norm(c, axis=1, keepdims=True)


def test_two_groups_of_environments():
    L, d, chi = 44, 8, 100
    c = random_product(np.random.default_rng(3), L, d)
    with Context(L, d, chi, mode="fp64") as ctx:
        ctx.upload(*M.product_state(c, 1))
        rho2, rho1 = ctx.two_point_rdms()
    site = np.einsum("si,sj->sij", c, c.conj())
    assert np.max(np.abs(rho1 - site)) < 1e-13
    for l1 in range(L):
        for l2 in range(l1 + 1, L):
            ref = np.kron(site[l1], site[l2])
            assert np.max(np.abs(rho2[l1, l2] - ref)) < 1e-13, (l1, l2)


def entangled(rng, L, d, chi, steps):
    H = rng.normal(size=(L - 1, d * d, d * d)) + 1j * rng.normal(size=(L - 1, d * d, d * d))
    H = 0.5 * (H + H.conj().transpose(0, 2, 1))
    return random_product(rng, L, d), M.construct_propagators(H, 0.2 / d), steps


@pytest.mark.parametrize("d,L,chi,steps", [(2, 9, 3, 2), (2, 14, 65, 6), (3, 8, 27, 3), (4, 8, 64, 3), (5, 6, 25, 2),
                                           (6, 5, 36, 2), (8, 5, 10, 2)])
@pytest.mark.parametrize("phase", [False, True])
def test_pairs_against_the_oracle(d, L, chi, steps, phase):
    rng = np.random.default_rng([d, L, chi])
    c, U, steps = entangled(rng, L, d, chi, steps)
    ph = rng.choice([-1.0, 1.0], d) if phase else None
    with Context(L, d, chi, mode="batched") as ctx:
        ctx.upload(*M.product_state(c, chi))
        ctx.set_gates(U)
        for _ in range(steps):
            ctx.trotter_step()
        rho2, rho1 = ctx.two_point_rdms(ph)
        gam, lam = ctx.download(chi)
    ref2, ref1 = two_point_rdms(gam, lam, ph)[:2]
    assert np.max(np.abs(rho1 - ref1)) < 1e-11
    for l1 in range(L):
        for l2 in range(l1 + 1, L):
            assert np.max(np.abs(rho2[l1, l2] - ref2[l1, l2])) < 1e-11, (l1, l2)


def test_ensemble_equals_its_chains():
    rng = np.random.default_rng(8)
    L, d, chi = 7, 2, 8
    sets = [entangled(rng, L, d, chi, 3) for _ in range(2)]
    single = []
    for c, U, steps in sets:
        with Context(L, d, chi, mode="batched") as ctx:
            ctx.upload(*M.product_state(c, chi))
            ctx.set_gates(U)
            for _ in range(steps):
                ctx.trotter_step()
            single.append((ctx.two_point_rdms(), ctx.download(chi)))
    with Ensemble(2, L, d, chi, mode="batched") as ens:
        ens.upload_chains(np.array([s[1][0] for s in single]), np.array([s[1][1] for s in single]))
        rho2, rho1 = ens.two_point_rdms()
    for r, ((ref2, ref1), _) in enumerate(single):
        assert np.max(np.abs(rho2[r] - ref2)) < 1e-13
        assert np.max(np.abs(rho1[r * L:(r + 1) * L] - ref1)) < 1e-13
