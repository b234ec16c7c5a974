"""The augmented-pencil kernels (every MFMA-named tile shape) on the launches
the tile-shape tests leave out: batches whose workgroups lie inside one
instance, cross from one to the next, or end partially filled, at the orders
where a workgroup holds several elements, and above p = 15, where the product
changes between the VALU and the MFMA form by form and velocity.  Both add the
same products in the same order, so every instance equals its solve alone bit
for bit, and constant velocities equal field reads."""
import numpy as np
import pytest

import dgk
from dgk import inputs

pytestmark = pytest.mark.gpu

# element counts whose sums fall on and between multiples of the elements per
# workgroup (64 at p = 1 down to 2 at p = 4)
BOXES = [(4, 4, 4), (3, 1, 1), (5, 3, 1), (2, 2, 2), (7, 1, 3), (1, 1, 1)]


@pytest.mark.parametrize("form,p", [(f, p) for f in ("HIP", "HIP_MP") for p in (2, 3, 4, 5, 7)])
def test_batch_workgroups_across_instances(form, p):
    rng = np.random.RandomState(p)
    inst = [dict(ne=ne, p=p, dt=2e-4 * (1 + k)) for k, ne in enumerate(BOXES)]
    vel = [tuple(rng.uniform(-1, 1, 3)) for _ in BOXES]
    for cand in range(len(dgk.tile_shapes(form, p))):
        # the run kernel does not take batches; the mixed form's VALU kernel takes
        # a batch's constant velocity unrounded, a solver's FP32 fields rounded
        if dgk.kernel_name(form, p, cand).startswith(("stage_run", "stage_f64_mp")):
            continue
        try:
            dgk.tile_select(form, p, cand)
            with dgk.Batch(form, inst) as b:
                for k in range(len(BOXES)):
                    b.init_gaussian(k, (0.3, 0.5, 0.6), 0.2, vel[k])
                b.step(3)
                got = [b.get_field(k) for k in range(len(BOXES))]
            for k, it in enumerate(inst):
                with dgk.Solver.structured(form, *it["ne"], p) as s:
                    s.init_gaussian((0.3, 0.5, 0.6), 0.2, vel[k])
                    s.step(it["dt"], 3)
                    assert np.array_equal(got[k], s.get_field(dgk.FIELD_Q)), (cand, k)
        finally:
            dgk.tile_select(form, p, -1)


@pytest.mark.parametrize("form,p", [("HIP", 16), ("HIP", 17), ("HIP_MP", 16), ("HIP_MP", 17),
                                    ("HIP_MP", 18), ("HIP_MP", 19)])
def test_valu_and_mfma_products_agree(monkeypatch, form, p):
    """Constant-velocity launches of the direction-by-direction shape run on the
    MFMA, the launches that read the same fields (FP64, mixed p >= 18) or the
    all-at-once shape on the VALU: the same bits."""
    ne = (2, 1, 3)
    q = inputs.random_fields(*ne, p, seed=60 + p)[0]
    const = [np.full_like(q, c) for c in (0.4, -0.3, 0.55)]
    got = []
    try:
        for cand in range(len(dgk.tile_shapes(form, p))):
            for env in ("1", "0"):
                monkeypatch.setenv("DGK_CVEL", env)
                dgk.tile_select(form, p, cand)
                with dgk.Solver.structured(form, *ne, p) as s:
                    s.set_fields(q, *const)
                    tend = s.cal_tend()
                    s.step(1e-5, 2)
                    got.append((tend, s.get_field(dgk.FIELD_Q)))
    finally:
        dgk.tile_select(form, p, -1)
    for a, b in got[1:]:
        assert np.array_equal(a, got[0][0]) and np.array_equal(b, got[0][1])
