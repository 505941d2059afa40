"""Schmidt values of a number-conserving evolution, against the record of an earlier build.

A disordered Fermi-Hubbard chain of 20 sites at chi = 100, ten steps and one shorter one, from a
number eigenstate.  The number blocks' values are cut at 1e-10, where rounding decides which states
stay, and values next to the cut move the others by up to 1e-8 over a few steps: a run is only
continued by a later build if the blocks are factorised with the same arithmetic.
golden/nc_fh_l20_chi100_lambdas.npz holds the propagators and the values that this library gave on
an MI355X with every pair visit of the Jacobi solved by cyclic sweeps and the blocks' QR panels
normed column by column; single passes move this chain by 1.1e-11.  The same operations in the same
order give the same bits; 1e-12 is the bound.
"""
import os

import numpy as np
import pytest

from tebd_amd import Context, models as M

pytestmark = pytest.mark.gpu

NUMBERS = np.array([0, 1, 1, 2], np.int32)


def test_values_are_those_of_the_record():
    with np.load(os.path.join(os.path.dirname(__file__), "golden", "nc_fh_l20_chi100_lambdas.npz")) as z:
        occ, warm, last, steps, lam = z["occ"], z["warm"], z["last"], int(z["steps"]), z["lam"]
    L, chi = occ.size, lam.shape[1]
    c = np.zeros((L, 4), np.complex128)
    c[np.arange(L), occ] = 1.0
    total = int(NUMBERS[occ].sum())
    print(f"[gpu] number-conserving chain, L = {L}, chi = {chi}", flush=True)
    with Context(L, 4, chi, mode="batched") as ctx:
        ctx.upload(*M.product_state(c, chi))
        ctx.set_gates(warm)
        ctx.set_conserved(NUMBERS, total, labels=M.product_labels(c, chi, NUMBERS, total))
        for _ in range(steps):
            ctx.trotter_step()
        ctx.set_gates(last)
        ctx.trotter_step()
        got = ctx.lambdas()
    assert np.max(np.abs(got - lam)) < 1e-12
