"""The mixed form's VALU kernel (its default at p = 1, a candidate up to p = 7) on
constant velocities: a box of a batch and a served request equal the same box on
a solver, bit for bit, also when another box of the batch has a varying wind and
the group reads the fields."""
import numpy as np
import pytest

import dgk
from dgk import inputs, serving

pytestmark = pytest.mark.gpu
CENTRE, SIGMA, VEL = (0.3, 0.5, 0.6), 0.2, (0.4, -0.3, 0.55)
BOXES = [(4, 3, 2), (3, 1, 2)]


def alone(ne, p, dt, nstep):
    with dgk.Solver.structured("HIP_MP", *ne, p) as s:
        s.init_gaussian(CENTRE, SIGMA, VEL)
        s.step(dt, nstep)
        return s.get_field(dgk.FIELD_Q)


@pytest.mark.parametrize("p", [1, 2, 4, 5, 7])
def test_batch_equals_solver(p):
    try:
        dgk.tile_select("HIP_MP", p, len(dgk.tile_shapes("HIP_MP", p)) - 1)
        assert dgk.kernel_name("HIP_MP", p, len(dgk.tile_shapes("HIP_MP", p)) - 1).startswith("stage_f64_mp<")
        ref = [alone(ne, p, 2e-3, 4) for ne in BOXES]
        for varying in (False, True):
            with dgk.Batch("HIP_MP", [dict(ne=ne, p=p, dt=2e-3) for ne in BOXES]) as b:
                for k in range(2):
                    b.init_gaussian(k, CENTRE, SIGMA, VEL)
                if varying:
                    b.set_field(1, dgk.FIELD_W, inputs.random_fields(*BOXES[1], p, seed=5)[3])
                b.step(4)
                assert np.array_equal(b.get_field(0), ref[0]), varying
                assert varying or np.array_equal(b.get_field(1), ref[1])
    finally:
        dgk.tile_select("HIP_MP", p, -1)


def test_served_request_equals_solver_at_p1():
    ne = (5, 4, 3)
    with serving.Server(64 << 20) as srv:
        out = np.empty((60, 8))
        srv.submit(dict(ne=ne, p=1, nstep=6, tol_class=1, vel=VEL, centre=CENTRE, sigma=SIGMA,
                        dt=2e-3), q_out=out)
        assert srv.wait(1)[0]["status"] == dgk.OK
    assert np.array_equal(out, alone(ne, 1, 2e-3, 6))
