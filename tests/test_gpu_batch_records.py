"""Workgroups of a batch that lie inside one instance (the geometry record read
as scalars) or cross into the next (per lane), at the orders where a workgroup
holds several elements, in both kinds of launch: constant velocities, and the
velocity fields, which the group reads when one instance's wind varies.  Every
instance equals its solve alone, bit for bit."""
import numpy as np
import pytest

import dgk
from dgk import inputs

pytestmark = pytest.mark.gpu

# element counts whose sums fall on, before and past multiples of the elements
# per workgroup (64, 32 and 16 at p = 1, 28, 14 and 7 at p = 2, ...)
BOXES = [(4, 4, 4), (3, 1, 1), (5, 3, 1), (2, 2, 2), (7, 1, 3), (1, 1, 1), (4, 4, 3), (31, 1, 1)]


@pytest.mark.parametrize("varying", [False, True])
@pytest.mark.parametrize("form,p", [(f, p) for f in ("HIP", "HIP_MP") for p in (1, 2, 3, 4)])
def test_instances_equal_their_solves(form, p, varying):
    rng = np.random.RandomState(p)
    inst = [dict(ne=ne, p=p, dt=2e-4 * (1 + k)) for k, ne in enumerate(BOXES)]
    vel = [tuple(rng.uniform(-1, 1, 3)) for _ in BOXES]
    wind = inputs.random_fields(*BOXES[4], p, seed=9, vel_scale=0.5)[1:]

    def fill(s, k, *at):
        s.init_gaussian(*at, (0.3, 0.5, 0.6), 0.2, vel[k])
        if varying and k == 4:
            for which, f in zip((dgk.FIELD_U, dgk.FIELD_V, dgk.FIELD_W), wind):
                s.set_field(*at, which, f)

    for cand in range(len(dgk.tile_shapes(form, p))):
        try:
            dgk.tile_select(form, p, cand)
            with dgk.Batch(form, inst) as b:
                for k in range(len(BOXES)):
                    fill(b, k, k)
                b.step(3)
                got = [b.get_field(k) for k in range(len(BOXES))]
            for k, it in enumerate(inst):
                with dgk.Solver.structured(form, *it["ne"], p) as s:
                    fill(s, k)
                    s.step(it["dt"], 3)
                    assert np.array_equal(got[k], s.get_field(dgk.FIELD_Q)), (cand, k)
        finally:
            dgk.tile_select(form, p, -1)
