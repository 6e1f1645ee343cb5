"""Into how many chunks the gated delta rule's long sequences are cut, where that was measured: the numbers within 4 parts in 100 of the fastest on 256
compute units (host code only)."""

import pytest

from beholdd.kernels import KernelSizes


@pytest.fixture(scope="module")
def lib():
    return KernelSizes(verbose_build=False).lib


@pytest.mark.parametrize("seqs,rows,heads,dim,vdim,fast", [
    (1, 4096, 128, 64, 64, [3]), (1, 2048, 128, 64, 64, [3]), (4, 1024, 32, 64, 64, [3]), (1, 2048, 16, 64, 64, [8, 12]), (1, 2048, 32, 128, 128, [3, 4]),
    (1, 2048, 16, 128, 128, [6, 8]), (1, 2048, 48, 128, 128, [3]), (1, 512, 32, 128, 128, [3, 4]), (1, 4096, 32, 128, 64, [4, 5, 8]), (1, 8192, 20, 96, 96, [8]),
    (1, 2048, 8, 256, 256, [2])])
def test_chunks_of_long_sequences(lib, seqs, rows, heads, dim, vdim, fast):
    chunk = lib.bh_delta_chunk_rows(seqs, rows, heads, dim, vdim)
    assert -(-rows // chunk) in fast and chunk % 16 == 0


@pytest.mark.parametrize("seqs,rows,heads,dim,vdim", [(1, 191, 1, 64, 64), (8, 2048, 64, 128, 128), (64, 4096, 64, 16, 16), (1, 4096, 4, 260, 64), (3, 1, 8, 64, 64)])
def test_sequences_that_are_walked_whole(lib, seqs, rows, heads, dim, vdim):
    assert lib.bh_delta_chunk_rows(seqs, rows, heads, dim, vdim) == rows
