"""Cutting one system's run in time (no GPU needed): the plan's shape."""

import pytest

from superspinsim_amd import _lib
from superspinsim_amd.generate_simulator import (
    MAX_CHUNK_DOUBLES, MAX_CHUNK_WAVES, time_chunks)


@pytest.mark.parametrize("n_out,fine,n,J,products,matrices,pairs", [
    (20, 300, 19, 5, 5, 6, True), (50, 20, 3, 5, 8, 6, True),
    (50, 20, 3, 5, 8, 6, False), (1, 997, 9, 2, 11, 2, False),
    (2000, 1, 64, 2, 11, 2, False), (10000, 100, 4, 2, 11, 2, True),
    (7, 1000, 49, 6, 30, 8, False), (1, 1000000, 2, 1, 11, 2, False)])
def test_chunks_cover_the_run(n_out, fine, n, J, products, matrices, pairs):
    split = time_chunks(n_out, fine, n, J, products, matrices, pairs)
    assert split is not None
    a, P, L, pack = split
    total = n_out * a
    assert fine % a == 0 and n % pack == 0 and pack * n <= _lib.MAX_N
    assert (P - 1) * L < total <= P * L and P > 1
    assert P * (n // pack) <= MAX_CHUNK_WAVES
    assert total * n * n <= MAX_CHUNK_DOUBLES
    assert not pairs or pack == 1 or n % 2 == 0


def test_short_and_wide_runs_stay_whole():
    assert time_chunks(1, 1, 9, 2, 11, 2) is None
    assert time_chunks(3, 2, 49, 2, 11, 2) is None
    assert time_chunks(1000, 100, 65, 2, 11, 2) is None
    assert time_chunks(10 ** 6, 100, 64, 2, 11, 2) is None
