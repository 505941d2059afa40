"""Bonds of more than 512 rows, whose Jacobi visits rotate the pairs within the column blocks too.

One Trotter step of a saturated Hubbard chain (bond matrices of 800 x 800) in one batch, whose
tasks lie on both sides of that bound, against the same step bond by bond.  Bound, fixed before
the first run: 1e-9 on every lambda and local occupation, as for all parity checks of evolved
states.
"""
import numpy as np
import pytest

from tebd_amd import Context, models as M

pytestmark = pytest.mark.gpu


def test_step_with_and_without_within_block_rotations():
    L, chi, dt = 96, 200, 0.05
    H = M.fermi_hubbard(L, 1.0, 4.0)
    U = M.construct_propagators(H, dt)
    with Context(L, 4, chi, mode="batched,learned") as ctx:
        ctx.upload(*M.product_state(M.neel(L, 4, 1, 2), chi))
        ctx.set_gates(U)
        for _ in range(16):
            ctx.trotter_step()
        start = ctx.download(chi)
        assert np.min(ctx.bond_dims()[10:-10]) == chi
    n = M.fermion_ops(2)[2]
    res = []
    for mode in ("batched", "fp64"):
        print(f"[gpu] within-block rotations, {mode}", flush=True)
        with Context(L, 4, chi, mode=mode) as ctx:
            if mode == "batched":
                ctx.set_lanes(1)
            ctx.upload(*start)
            ctx.set_gates(U)
            ctx.trotter_step()
            res.append((ctx.download(chi)[1], ctx.one_site_expval(n)))
    assert np.max(np.abs(res[0][0] - res[1][0])) < 1e-9
    assert np.max(np.abs(np.asarray(res[0][1]) - np.asarray(res[1][1]))) < 1e-9
