"""dgk_minmax (one launch, the last block folds) at the sizes where its blocks
change: one value short of and past a block's 2048, exactly the most blocks,
past them; called again and again on one handle, with extremes at the ends,
infinities, and NaN (ignored, as fmin and fmax do)."""
import numpy as np
import pytest

import dgk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ne", [1, 255, 256, 257, 4099, 262144, 262151])
def test_minmax_sizes(ne):
    rng = np.random.RandomState(ne)
    with dgk.Solver.structured("HIP", ne, 1, 1, 1) as s:
        for k in range(4):
            q = rng.uniform(-1.0, 1.0, (ne, 8))
            if k == 1:
                q[0, 0], q[-1, -1] = -5.0, 7.0
            elif k == 2:
                q[-1, -1], q[0, 0] = -np.inf, np.inf
            elif k == 3:
                q[ne // 2, 3] = np.nan
            s.set_field(dgk.FIELD_Q, q)
            for _ in range(3):
                assert s.minmax() == (np.nanmin(q), np.nanmax(q))


def test_minmax_all_nan():
    with dgk.Solver.structured("HIP", 3, 1, 1, 1) as s:
        s.set_field(dgk.FIELD_Q, np.full((3, 8), np.nan))
        assert s.minmax() == (np.inf, -np.inf)
