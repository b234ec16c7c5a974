"""The pencil kernel (the axis-aligned register form, candidate 1 of "HIP") on
the launches the tile-shape tests leave out: a resolved face-node table, a
geometry record per element, and both with a partial last workgroup.  It
performs the staged kernel's operations in the same order, so the bits are
equal; the oracle bounds are the FP64 ones."""
import numpy as np
import pytest

import dgk
import oracle
from dgk import inputs

pytestmark = pytest.mark.gpu


def mesh(ne, p, twisted, records):
    m = oracle.Mesh(*ne, p)
    if records:
        scale = 1.0 + 0.25 * np.arange(m.Ne)
        m.Escale = np.ascontiguousarray(m.Escale * scale[None, :, None])
        m.Fscale = np.ascontiguousarray(m.Fscale * scale[:, None])
    if twisted:
        perm = np.arange(m.Nfp).reshape(m.Nq, m.Nq).T.reshape(-1)
        VP = m.VMapP.copy()
        for e in range(m.Ne):
            for f in (4, 5):
                seg = VP[e, f * m.Nfp:(f + 1) * m.Nfp].copy()
                VP[e, f * m.Nfp:(f + 1) * m.Nfp] = seg[perm]
        m.VMapP = VP
    return m


@pytest.mark.parametrize("twisted,records", [(True, False), (False, True), (True, True)])
@pytest.mark.parametrize("p", [1, 2, 3, 4, 5, 7, 8, 12, 15])
def test_pencil_equals_staged(p, twisted, records):
    ne = (3, 2, 3) if p <= 7 else (2, 1, 2)
    m = mesh(ne, p, twisted, records)
    q, u, v, w = inputs.random_fields(*ne, p, seed=900 + p, vel_scale=0.7)
    ref = m.cal_tend(m.field(q), m.field(u), m.field(v), m.field(w))
    got = []
    try:
        for cand in (0, 1):
            dgk.tile_select("HIP", p, cand)
            with dgk.Solver.create("HIP", m.Nq, m.Ne, m.NeA, m.NhaloNode, m.D, m.Lift, m.VMapM,
                                   m.VMapP, m.halo_src_map, m.normal_fn, m.Escale, m.Fscale) as s:
                s.set_fields(q, u, v, w)
                tend = s.cal_tend()
                s.step(1e-4, 2)
                got.append((tend, s.get_field(dgk.FIELD_Q)))
    finally:
        dgk.tile_select("HIP", p, -1)
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
    assert np.abs(got[1][0] - ref).max() <= 1e-13 * np.abs(ref).max()
