"""The column selection of the pivoted-QR panel, against LAPACK.

theta has only `live` non-zero rows and columns (of norms over five decades); a panel that took
an empty column while a live one is left would end the factorisation there and lose its Schmidt
values.  Column counts lie on both sides of the blocks of 64 that the selection ranks within,
the live columns are the last ones, all in one block, or spread, and their number and the last
panel's width take whole and broken panels of 16.

Tolerance, fixed before the first run: as for any backward stable SVD of a theta of norm 1 with
a stopping bound of 1e-13 per column pair, 1e-12 on lambda.
"""
import numpy as np
import pytest

from tebd_amd import Context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,chil,chir,live,where", [
    (2, 32, 32, 1, "last"), (2, 32, 32, 64, "last"), (2, 35, 33, 17, "last"), (2, 33, 50, 16, "one"), (2, 64, 64, 31, "spread"),
    (3, 43, 43, 33, "one"), (2, 100, 97, 48, "spread"), (2, 129, 129, 20, "last"), (4, 65, 64, 75, "spread"),
    (2, 256, 260, 18, "one")])
def test_live_columns_are_found(d, chil, chir, live, where):
    rng = np.random.default_rng([d, chil, chir, live])
    m, n = d * chil, d * chir

    def pick(size):
        if where == "last":
            return np.arange(size - live, size)
        if where == "one":
            return 64 + rng.permutation(min(64, size - 64))[:live] if size >= 64 + live else rng.permutation(size)[:live]
        return rng.permutation(size)[:live]

    rows, cols = pick(m), pick(n)
    left, right = np.zeros((m, live), np.complex128), np.zeros((live, n), np.complex128)
    left[rows] = np.linalg.qr(rng.normal(size=(live, live)) + 1j * rng.normal(size=(live, live)))[0]
    right[:, cols] = np.linalg.qr(rng.normal(size=(live, live)) + 1j * rng.normal(size=(live, live)))[0]
    lc = np.sort(10.0 ** rng.uniform(-5, 0, live))[::-1]
    lc /= np.linalg.norm(lc)
    chi = max(chil, chir, live)
    gam = np.zeros((2, chi, d, chi), np.complex128)                      # site, b, i, a
    gam[0, :live, :, :chil] = left.reshape(chil, d, live).transpose(2, 1, 0)
    gam[1, :chir, :, :live] = right.reshape(live, d, chir).transpose(2, 1, 0)
    lams = np.zeros((3, chi))
    lams[0, :chil] = 1.0
    lams[1, :live] = lc
    lams[2, :chir] = 1.0

    print(f"[gpu] select {m} x {n}, {live} live, {where}", flush=True)
    with Context(2, d, chi, mode="fp64") as ctx:
        ctx.upload(gam, lams)
        ctx.two_site_op(1, np.eye(d * d, dtype=np.complex128))
        _, l = ctx.download(chi)
    ref = np.zeros(chi)
    ref[:live] = lc
    assert np.max(np.abs(l[1] - ref)) < 1e-12
