"""Bonds without a side of 64: one launch for the whole SVD, or sweep by sweep beside larger bonds.

A bond of at most 32 columns is solved in one launch when every bond of its batch is such a bond, else
sweep by sweep with the others.  Bond by bond every one of them is alone; batched, a half-sweep holds
both kinds (chi = 24 and 20: up to 48 and 60 columns) or only the first (chi = 8 and 10).  Both routes
do the same operations in the same order: equal bits after several steps, with bonds that grow from
one kind into the other.
"""
import numpy as np
import pytest

from tebd_amd import Context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,L,chi", [(2, 12, 24), (3, 9, 20), (2, 9, 8), (3, 7, 10)])
def test_both_routes_give_the_same_bits(d, L, chi):
    rng = np.random.default_rng([d, L, chi])
    U = np.array([np.linalg.qr(rng.normal(size=(d * d, d * d)) + 1j * rng.normal(size=(d * d, d * d)))[0] for _ in range(L - 1)])
    c = rng.normal(size=(L, d)) + 1j * rng.normal(size=(L, d))
    gam = (c / np.linalg.norm(c, axis=1, keepdims=True)).reshape(L, 1, d, 1)
    res = []
    for mode in ("fp64", "batched"):
        print(f"[gpu] {L} sites of d = {d}, chi = {chi}, {mode}", flush=True)
        with Context(L, d, chi, mode=mode) as ctx:
            ctx.upload(gam, np.ones((L + 1, 1)))
            ctx.set_gates(U)
            for _ in range(5):
                ctx.trotter_step()
            res.append(ctx.download(chi))
    assert np.array_equal(res[0][1], res[1][1])
    assert np.array_equal(res[0][0], res[1][0])
