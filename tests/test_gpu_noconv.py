"""A bond update whose SVD does not converge leaves the state as it was.

An operator of 1e78 makes the Gram matrices of theta overflow in their squares, so no pair of columns
of the small solve is ever found orthogonal.  The call reports TEBD_ERR_NOCONV (-5); Gammas, lambdas
and bond dimensions are those from before it, and the next update of the same context is right.
"""
import numpy as np
import pytest

from tebd_amd import Context, TEBDError

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["fp64", "batched"])
def test_state_survives_a_failed_update(mode):
    n = 16
    rng = np.random.default_rng(n)

    def cplx(*shape):
        return rng.normal(size=shape) + 1j * rng.normal(size=shape)

    gam = np.array([cplx(n, 2, n), cplx(n, 2, n)])
    lam = np.repeat(np.sort(rng.uniform(0.1, 1.0, n))[::-1][None], 3, axis=0)
    with Context(2, 2, n, mode=mode) as ctx, Context(2, 2, n, mode=mode) as ref:
        ctx.upload(gam, lam)
        ref.upload(gam, lam)
        before = ctx.download(n)
        with pytest.raises(TEBDError) as err:
            ctx.two_site_op(1, np.eye(4) * 1e78)
        assert "converge" in str(err.value)
        after = ctx.download(n)
        assert np.array_equal(before[0], after[0]) and np.array_equal(before[1], after[1])
        for c in (ctx, ref):
            c.two_site_op(1, np.eye(4))
        assert np.array_equal(ctx.lambdas(), ref.lambdas())
