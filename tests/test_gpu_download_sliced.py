"""Sliced downloads on the device: with the pinned chunks made first, every size
of 4 MiB and more goes through them, at the sizes where chunks and slices change."""
import numpy as np
import pytest

import dgk

pytestmark = pytest.mark.gpu


def field(s):
    n = s.Ne * s.Np
    return (np.arange(n, dtype=np.float64) * 1.25 - 7.0).reshape(s.Ne, s.Np)


@pytest.fixture(scope="module")
def chunks():
    with dgk.Solver.structured("HIP", 49, 48, 50, 3) as s:  # 60 MB: the first download makes them
        q = field(s)
        s.set_field(dgk.FIELD_Q, q)
        assert np.array_equal(s.get_field(dgk.FIELD_Q), q)
        yield s


# elements of p = 3 (512 bytes each): 4 MiB, one element more, either side of
# 8 MiB (a chunk per slice), 16 MiB and a bit, odd ones
@pytest.mark.parametrize("ne", [(8192, 1, 1), (8193, 1, 1), (5461, 3, 1), (16384, 1, 1),
                                (16393, 1, 1), (32771, 1, 1), (331, 7, 13)])
def test_every_large_size(chunks, ne):
    with dgk.Solver.structured("HIP", *ne, 3) as s:
        q = field(s)
        s.set_field(dgk.FIELD_Q, q)
        for _ in range(3):
            assert np.array_equal(s.get_field(dgk.FIELD_Q), q)
        assert np.array_equal(s.get_field(dgk.FIELD_Q, with_halo=True)[: s.Ne], q)
