"""The scratch memory that the byte plan counts for the recurrences covers every smaller step, not only the largest
one: a step of one long sequence may take more than one of as many sequences as the engine holds."""

import ctypes
import random

import pytest

from beholdd.kernels import KernelSizes


@pytest.fixture(scope="module")
def sizes():
    return KernelSizes(verbose_build=False)


def lightning_takes(lib, seqs, rows, longest, heads, dim, vdim, stride):
    """Bytes that `lightning_scan` asks for (`stride` 0: rows that go as products where that is faster, 1: rows that cannot)."""
    floats = lib.bh_lightning_products_scratch(seqs, rows, longest, heads, dim, vdim, stride, 0, 0, 0)
    if not floats:
        cut = ctypes.c_int(0)
        chunks = lib.bh_lightning_chunks(seqs, rows, longest, heads, vdim, ctypes.byref(cut))
        floats = seqs * chunks * heads * dim * vdim if chunks > 1 else 0
    return floats * 4


def ssm_takes(lib, seqs, rows, longest, heads, vdim, n_state, stride):
    floats = lib.bh_ssm_products_scratch(seqs, rows, longest, heads, vdim, n_state, 1, stride)
    if not floats and lib.bh_ssm_fast_takes(vdim, n_state):
        chunks = -(-longest // lib.bh_ssm_chunk_rows(seqs, longest, heads))
        floats = seqs * chunks * heads * (n_state * vdim + 1) + rows * heads if chunks > 1 else 0
    return floats * 4


@pytest.mark.parametrize("seqs,rows,longest,heads,dim,vdim", [
    (64, 2048, 2048, 256, 128, 64), (64, 512, 512, 128, 128, 64), (16, 8192, 4096, 32, 128, 128), (1, 300, 300, 8, 256, 256), (500, 700, 700, 4, 64, 48),
    (3, 129, 129, 1, 64, 16), (64, 64, 1, 32, 128, 128), (8, 127, 127, 3, 48, 24), (64, 4096, 512, 16, 96, 64)])
def test_a_plan_covers_every_step_of_its_sizes(sizes, seqs, rows, longest, heads, dim, vdim):
    rng = random.Random(rows + heads)
    planned = (sizes.lightning_chunk_bytes(seqs, rows, longest, heads, dim, vdim), sizes.ssm_chunk_bytes(seqs, rows, longest, heads, vdim, dim))
    steps = [(n, min(rows, r)) for n in (1, 2, 3, 7, seqs // 2, seqs) for r in (rows, rows // 2, 128, 64, n) if 1 <= n <= min(seqs, r)]
    steps += [(n, rng.randint(n, rows)) for n in (rng.randint(1, min(seqs, rows)) for _ in range(300))]
    for n, r in steps:
        for most in {min(longest, r - n + 1), -(-r // n), rng.randint(-(-r // n), max(min(longest, r - n + 1), -(-r // n)))}:
            if most > longest:
                continue
            for stride in (0, 1):
                assert lightning_takes(sizes.lib, n, r, most, heads, dim, vdim, stride) <= planned[0], (n, r, most, stride)
                assert ssm_takes(sizes.lib, n, r, most, heads, vdim, dim, stride) <= planned[1], (n, r, most, stride)
    if longest == 1:
        assert planned == (0, 0)      # captured decode steps take none


def delta_takes(lib, seqs, rows, longest, heads, dim, vdim):
    chunk = lib.bh_delta_chunk_rows(seqs, longest, heads, dim, vdim)
    return (seqs * -(-longest // chunk) * heads * dim * (vdim + dim) + rows * heads * dim) * 4 if chunk < longest else 0


def gla_takes(lib, seqs, rows, longest, heads, dim, vdim):
    chunk = lib.bh_gla_chunk_rows(seqs, longest, heads, dim, vdim)
    return (seqs * -(-longest // chunk) * heads * dim * (vdim + 1) + rows * heads * dim) * 4 if chunk < longest else 0


# one sequence of many heads, many of few; heads of every kind of walk; sequences shorter than the step; steps that are never cut
@pytest.mark.parametrize("seqs,rows,longest,heads,dim,vdim", [
    (4, 8192, 8192, 8, 128, 128), (8, 8192, 8192, 32, 128, 128), (64, 2048, 2048, 32, 128, 128), (16, 8192, 4096, 16, 128, 128), (1, 300, 300, 8, 256, 256),
    (8, 4096, 4096, 96, 64, 64), (64, 4096, 512, 16, 96, 64), (2, 8192, 8192, 4, 256, 250), (32, 16384, 8192, 4, 64, 64), (8, 1000, 1000, 32, 32, 32), (300, 700, 700, 2, 20, 48),
    (4, 6000, 6000, 3, 300, 64), (64, 64, 1, 32, 128, 128)])
def test_a_plan_covers_every_step_of_the_recurrences_that_are_joined(sizes, seqs, rows, longest, heads, dim, vdim):
    rng = random.Random(rows + heads)
    plans = sizes.delta_chunk_bytes(seqs, rows, longest, heads, dim, vdim), sizes.gla_chunk_bytes(seqs, rows, longest, heads, dim, vdim)
    largest = [0, 0]
    for n in range(1, seqs + 1):
        most = min(longest, rows - n + 1)
        for m in {most, max(most // 2, 1), *(rng.randint(1, most) for _ in range(3000 // seqs + 20)), *range(128, most + 1, 64)}:
            for at, takes in enumerate((delta_takes, gla_takes)):
                taken = takes(sizes.lib, n, min(rows, n * m), m, heads, dim, vdim)
                assert taken <= plans[at], (n, m, at)
                largest[at] = max(largest[at], taken)
    assert all(plan <= 1.65 * most for plan, most in zip(plans, largest))      # and not much more: a limit on memory refuses by it
