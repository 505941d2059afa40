"""All-pairs density matrices and expectation values while device memory is short.

Memory is held until 700 MiB are left.  The environments of 24 sites of d = 8 with room for chi = 100
take 2.5 GB in one group, one alone 100 MB: the call has to do with smaller groups and give the same
matrices.  One environment with room for chi = 300 takes 920 MB: that call fails, leaves nothing
allocated, and succeeds on the same context once memory is there again, as do the other calls.

On a product state every pair's matrix is the product of the two sites' own, which is exact: 1e-13.
"""
import ctypes

import numpy as np
import pytest

from tebd_amd import Context, TEBDError, models as M

pytestmark = pytest.mark.gpu

MIB = 1 << 20


class Held:
    """All but `left` bytes of the device's memory, from the HIP runtime that the library uses."""

    def __init__(self, left):
        self.hip = ctypes.CDLL("libamdhip64.so.7", mode=ctypes.RTLD_GLOBAL)
        self.hip.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
        self.hip.hipFree.argtypes = [ctypes.c_void_p]
        self.held = []
        while self.free() > left + 4 * MIB:  # the first allocations change what the runtime itself reserves
            p = ctypes.c_void_p()
            assert len(self.held) < 8 and self.hip.hipMalloc(ctypes.byref(p), self.free() - left) == 0
            self.held.append(p)

    def free(self):
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert self.hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        for p in self.held:
            assert self.hip.hipFree(p) == 0


def product(L, d):
    rng = np.random.default_rng([L, d])
    c = rng.normal(size=(L, d)) + 1j * rng.normal(size=(L, d))
    return c / np.linalg.norm(c, axis=1, keepdims=True)


def check(c, rho2):
    site = np.einsum("si,sj->sij", c, c.conj())
    for l1 in range(len(c)):
        for l2 in range(l1 + 1, len(c)):
            assert np.max(np.abs(rho2[l1, l2] - np.kron(site[l1], site[l2]))) < 1e-13


def test_smaller_groups_when_memory_is_short():
    L, d, chi = 24, 8, 100
    c = product(L, d)
    with Context(L, d, chi, mode="fp64") as ctx:
        ctx.upload(*M.product_state(c, 1))
        ctx.sync()
        print("[gpu] density matrices in 700 MiB", flush=True)
        with Held(700 * MIB):
            rho2, _ = ctx.two_point_rdms()
            vals = ctx.expval_two_site(np.repeat(np.eye(d * d)[None], L - 1, axis=0))
    check(c, rho2)
    assert np.max(np.abs(vals - 1.0)) < 1e-13


def test_a_failed_call_leaves_nothing_allocated():
    L, d, chi = 4, 8, 300
    c = product(L, d)
    ops = np.repeat(np.eye(d * d)[None], L - 1, axis=0)
    with Context(L, d, chi, mode="fp64") as ctx:
        ctx.upload(*M.product_state(c, 1))
        ctx.expval_two_site(ops)
        ctx.sync()
        print("[gpu] density matrices that do not fit 700 MiB", flush=True)
        with Held(700 * MIB) as held:
            free = held.free()
            for _ in range(3):
                with pytest.raises(TEBDError):
                    ctx.two_point_rdms()
            assert held.free() == free
            assert np.max(np.abs(ctx.expval_two_site(ops) - 1.0)) < 1e-13
        rho2, _ = ctx.two_point_rdms()
    check(c, rho2)
