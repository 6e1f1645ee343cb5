"""Which form the recurrences with a scalar decay take, on both sides of each line, at the compute-unit count that the library assumes
where there is no GPU (256): the walk row by row, or products of matrices over chunks of 64 rows.  Both give the same numbers."""

import pytest

from beholdd.kernels import KernelSizes


@pytest.fixture(scope="module")
def lib():
    return KernelSizes(verbose_build=False).lib


@pytest.mark.parametrize("seqs,rows,longest,heads,dim,vdim,products", [
    (1, 127, 127, 16, 128, 128, False), (1, 128, 128, 16, 128, 128, True), (200, 200, 200, 16, 128, 128, False),
    (1, 256, 256, 4, 256, 256, False), (1, 320, 320, 4, 256, 256, True), (1, 256, 256, 8, 64, 256, False), (1, 320, 320, 8, 64, 256, True),
    (1, 256, 256, 4, 256, 128, True), (8, 137, 130, 1, 256, 256, False),
    (64, 191, 128, 32, 128, 128, True), (217, 344, 128, 32, 128, 128, True), (218, 345, 128, 32, 128, 128, False), (512, 811, 300, 64, 128, 128, False),
    (281, 408, 128, 16, 64, 64, True), (282, 409, 128, 16, 64, 64, False), (512, 639, 128, 1, 128, 128, True), (512, 639, 128, 32, 192, 128, True),
    (115, 242, 128, 128, 64, 16, True), (116, 243, 128, 128, 64, 16, False)])
def test_lightning(lib, seqs, rows, longest, heads, dim, vdim, products):
    stride = 2 * heads * (dim + vdim)
    assert (lib.bh_lightning_products_scratch(seqs, rows, longest, heads, dim, vdim, stride, 0, heads * dim, 2 * heads * dim) > 0) == products


@pytest.mark.parametrize("seqs,rows,longest,heads,vdim,n_state,products", [
    (1, 63, 63, 32, 64, 128, False), (1, 64, 64, 32, 64, 128, True), (100, 100, 100, 8, 64, 128, False), (8, 512, 64, 64, 64, 64, True),
    (8, 512, 64, 64, 32, 64, False), (7, 448, 64, 64, 32, 64, True), (8, 520, 65, 8, 32, 64, True), (8, 512, 64, 128, 64, 128, False)])
def test_state_space(lib, seqs, rows, longest, heads, vdim, n_state, products):
    assert (lib.bh_ssm_products_scratch(seqs, rows, longest, heads, vdim, n_state, 1, heads * vdim + 2 * n_state) > 0) == products
