"""The mixed form at p = 13..15 runs launches of few elements (256, with a
constant velocity 512) on the MFMA and larger ones on the VALU, the same sums in
the same order: a box alone, on the first, equals the same box in a batch that is
large enough for the second, bit for bit.  Either side of the line both agree
with the oracle on every kind of mesh (the form's bound, 1e-5 relative L2)."""
import numpy as np
import pytest

import dgk
import oracle
from dgk import inputs

pytestmark = pytest.mark.gpu
TOL = 1e-5


@pytest.mark.parametrize("wind", ["constant", "varying"])
@pytest.mark.parametrize("p", [13, 14, 15])
def test_box_alone_equals_box_in_a_large_batch(p, wind):
    boxes = [(3, 1, 2), (9, 9, 7), (5, 3, 4)]
    vel = [(0.4, -0.3, 0.55), (-0.7, 0.2, 0.1), (0.3, 0.9, -0.2)]
    fields = [inputs.random_fields(*ne, p, seed=20 + k, vel_scale=0.5)[1:] for k, ne in enumerate(boxes)]

    def fill(s, k, *at):
        s.init_gaussian(*at, (0.3, 0.5, 0.6), 0.2, vel[k])
        if wind == "varying":
            for which, f in zip((dgk.FIELD_U, dgk.FIELD_V, dgk.FIELD_W), fields[k]):
                s.set_field(*at, which, f)

    try:
        for cand in range(len(dgk.tile_shapes("HIP_MP", p))):
            dgk.tile_select("HIP_MP", p, cand)
            with dgk.Batch("HIP_MP", [dict(ne=ne, p=p, dt=1e-4) for ne in boxes]) as b:
                for k in range(3):
                    fill(b, k, k)
                b.step(3)
                for k in (0, 2):
                    with dgk.Solver.structured("HIP_MP", *boxes[k], p) as s:
                        fill(s, k)
                        s.step(1e-4, 3)
                        assert np.array_equal(s.get_field(dgk.FIELD_Q), b.get_field(k)), (cand, k)
    finally:
        dgk.tile_select("HIP_MP", p, -1)


@pytest.mark.parametrize("mesh", ["box", "records", "tilted", "twisted", "constant"])
@pytest.mark.parametrize("ne", [(8, 8, 4), (257, 1, 1), (8, 8, 8), (19, 9, 3)])
@pytest.mark.parametrize("p", [13, 15])
def test_both_sides_of_the_line_agree_with_the_oracle(p, ne, mesh):
    m = oracle.Mesh(*ne, p)
    if mesh == "records":
        scale = 1.0 + 0.25 * (np.arange(m.Ne) % 7)
        m.Escale = np.ascontiguousarray(m.Escale * scale[None, :, None])
        m.Fscale = np.ascontiguousarray(m.Fscale * scale[:, None])
    elif mesh == "tilted":
        m.normal_fn = np.ascontiguousarray(m.normal_fn + 0.05)
    elif mesh == "twisted":
        perm = np.arange(m.Nfp).reshape(m.Nq, m.Nq).T.reshape(-1)
        VP = m.VMapP.copy()
        for f in (4, 5):
            VP[:, f * m.Nfp:(f + 1) * m.Nfp] = VP[:, f * m.Nfp:(f + 1) * m.Nfp][:, perm]
        m.VMapP = VP
    q, u, v, w = inputs.random_fields(*ne, p, seed=400 + p, vel_scale=0.7)
    if mesh == "constant":
        u, v, w = (np.full_like(q, c) for c in (0.4, -0.3, 0.55))
    ref = m.cal_tend(m.field(q), m.field(u), m.field(v), m.field(w))
    with dgk.Solver.create("HIP_MP", m.Nq, m.Ne, m.NeA, m.NhaloNode, m.D, m.Lift, m.VMapM,
                           m.VMapP, m.halo_src_map, m.normal_fn, m.Escale, m.Fscale) as s:
        s.set_fields(q, u, v, w)
        got = s.cal_tend()
    assert np.linalg.norm(got - ref) <= TOL * np.linalg.norm(ref)
