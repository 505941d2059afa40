"""A bond's result does not depend on its batch where the QR of the batch's bonds takes different forms.

A chain of 7 sites of d = 8 at chi = 136: each half-sweep updates a bond of 512 x 8 (panels in
registers) together with bonds of 1088 rows (panels through global memory).  One step bond by bond and
one with all bonds of a half-sweep in a batch do the same operations on every bond: equal bits.
"""
import numpy as np
import pytest

from tebd_amd import Context

pytestmark = pytest.mark.gpu


def test_bonds_of_more_and_of_less_than_1024_rows():
    L, d, chi = 7, 8, 136
    rng = np.random.default_rng(L)
    dims = [min(chi, d ** min(b, L - b)) for b in range(L + 1)]
    gam = np.zeros((L, chi, d, chi), np.complex128)                      # site, b, i, a
    lam = np.zeros((L + 1, chi))
    for s in range(L):
        shape = (dims[s + 1], d, dims[s])
        gam[s, :dims[s + 1], :, :dims[s]] = rng.normal(size=shape) + 1j * rng.normal(size=shape)
    for b, n in enumerate(dims):
        v = np.sort(10.0 ** rng.uniform(-3, 0, n))[::-1]
        lam[b, :n] = v / np.linalg.norm(v)
    U = np.array([np.linalg.qr(rng.normal(size=(d * d, d * d)) + 1j * rng.normal(size=(d * d, d * d)))[0] for _ in range(L - 1)])
    res = []
    for mode in ("fp64", "batched"):
        print(f"[gpu] 7 sites of d = 8, chi = 136, {mode}", flush=True)
        with Context(L, d, chi, mode=mode) as ctx:
            ctx.set_lanes(1)
            ctx.upload(gam, lam)
            ctx.set_gates(U)
            ctx.trotter_step()
            res.append(ctx.download(chi))
    assert np.array_equal(res[0][1], res[1][1])
    assert np.array_equal(res[0][0], res[1][0])
