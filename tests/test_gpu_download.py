"""Downloads at the sizes where they change their way (plain below 4 MiB, sliced
over several threads above, once enough has been asked for), with remainders of
a chunk and of a slice, and from two threads at once."""
import threading

import numpy as np
import pytest

import dgk

pytestmark = pytest.mark.gpu

# elements of p = 3 (512 bytes each): around 4 MiB, 8 MiB + a bit, an odd size,
# and about 60 MB
SIZES = [(8191, 1, 1), (8192, 1, 1), (8193, 2, 1), (331, 7, 13), (49, 48, 50)]


def field(s):
    n = s.Ne * s.Np
    return (np.arange(n, dtype=np.float64) * 1.25 - 7.0).reshape(s.Ne, s.Np)


@pytest.mark.parametrize("ne", SIZES)
def test_download_returns_what_was_uploaded(ne):
    with dgk.Solver.structured("HIP", *ne, 3) as s:
        q = field(s)
        s.set_field(dgk.FIELD_Q, q)
        for _ in range(4):
            assert np.array_equal(s.get_field(dgk.FIELD_Q), q)
        assert np.array_equal(s.get_field(dgk.FIELD_Q, with_halo=True)[: s.Ne], q)


def test_downloads_from_two_threads():
    with dgk.Solver.structured("HIP", 48, 50, 49, 3) as keep:
        keep.set_field(dgk.FIELD_Q, field(keep))
        bad = []

        def work(k):
            with dgk.Solver.structured("HIP", 40 + k, 41, 39, 3) as s:
                q = field(s) + k
                s.set_field(dgk.FIELD_Q, q)
                for _ in range(6):
                    if not np.array_equal(s.get_field(dgk.FIELD_Q), q):
                        bad.append(k)

        t = [threading.Thread(target=work, args=(k,)) for k in range(2)]
        for x in t:
            x.start()
        for x in t:
            x.join()
        assert not bad
        assert np.array_equal(keep.get_field(dgk.FIELD_Q), field(keep))
