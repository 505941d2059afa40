"""The bond SVD on both sides of 512 rows, where a pair visit of the Jacobi goes from one pass of
rotations to whole cyclic sweeps, against LAPACK.

The check, its inputs' construction and its tolerances (1e-12 on lambda, 1e-11 on the product) are
those of test_gpu_svd_sizes: random graded site tensors, a random unitary operator, nothing
truncated.  Rows here are the smaller side of theta after the QR: 510 to 520 around the bound, one
block column beyond it, and 1024, at ranks that fill the bond and ranks that do not.
"""
import pytest

from test_gpu_svd_sizes import test_svd_of_every_kernel_shape as check_svd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,chil,chic,chir", [(2, 255, 140, 270), (2, 256, 128, 256), (2, 257, 150, 256), (2, 257, 129, 260),
                                              (4, 130, 20, 136), (4, 260, 64, 256)])
def test_svd_around_the_row_bound(d, chil, chic, chir):
    check_svd(d, chil, chic, chir)
