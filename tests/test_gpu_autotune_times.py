"""The autotuner times the launches that a step makes: its figure for the tile
shape that it keeps agrees with the step's own time per launch.  With the input
standing in for the RK base too (one of three streams not read) it reported 53 us
at FP64 p = 7 where the step took 68."""
import pytest

import dgk

pytestmark = pytest.mark.gpu

VEL = (0.3, -0.7, 0.5)
# timings of one kernel differ by 3%, the faults below by 20% and more; each
# figure is the least of three and a pair that disagrees is measured again, since
# something else may have held the device meanwhile
WITHIN = 0.10
ATTEMPTS = 3


def agree(pair):
    seen = []
    for _ in range(ATTEMPTS):
        tuned, step = pair()
        seen.append((tuned, step))
        if abs(tuned - step) < WITHIN * step:
            return
    raise AssertionError(seen)


@pytest.mark.parametrize("form,p,ne", [("HIP", 7, 32), ("HIP", 3, 64), ("HIP_MP", 7, 32)])
def test_solver_times_are_the_steps(form, p, ne):
    with dgk.Solver.structured(form, ne, ne, ne, p) as s:
        s.init_gaussian((0.3, 0.4, 0.5), 0.1, VEL)
        s.step(1e-5, 30)
        before = s.get_field(dgk.FIELD_Q)

        def tuned():
            runs = [s.autotune(60) for _ in range(3)]
            best = runs[-1]["best"]
            return min(r["us_per_launch"][best] for r in runs)

        def step():
            s.timer_reset()
            s.set_kernel_timing(True)
            s.step(1e-5, 40)
            s.synchronize()
            s.set_kernel_timing(False)
            seconds, n = s.timers()["Stage (fused)"]
            return 1e6 * seconds / n

        tuned()
        assert (s.get_field(dgk.FIELD_Q) == before).all()
        agree(lambda: (tuned(), min(step() for _ in range(3))))


@pytest.mark.parametrize("form,p,ne", [("HIP_MP", 2, 85), ("HIP", 3, 64), ("HIP", 7, 32)])
def test_batch_times_are_the_steps(form, p, ne):
    """A batch's launches read a workgroup's geometry record as scalars; timed as
    a solver's launches they took the per-lane reads (mixed p = 2, 125 against
    106 us in the step)."""
    with dgk.Batch(form, [dict(ne=(ne, ne, ne), p=p, dt=1e-5)]) as b:
        b.init_gaussian(0, (0.3, 0.4, 0.5), 0.1, VEL)
        b.step(20)
        b.synchronize()
        before = b.get_field(0)

        def tuned():
            runs = [b.autotune(reps=60)[0] for _ in range(3)]
            return min(r["us_per_launch"] for r in runs if r["candidate"] == runs[-1]["candidate"])

        def step():
            b.synchronize()
            b.timer()
            b.step(40)
            seconds, _ = b.timer()
            return 1e6 * seconds / 120

        tuned()
        assert (b.get_field(0) == before).all()

        def pair():
            t = tuned()
            b.step(20)
            return t, min(step() for _ in range(3))

        agree(pair)
