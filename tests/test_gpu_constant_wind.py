"""Solvers whose velocity fields hold one value each run the stage kernels
that read the wind from the geometry record; those results equal, bit for bit,
the launches that read the fields (DGK_CVEL=0 keeps them), whichever way the
constant fields arrived, and a varying field given later is read again."""
import numpy as np
import pytest

import dgk
import oracle
from dgk import inputs

pytestmark = pytest.mark.gpu
VEL = (0.4, -0.3, 0.55)


def results(s, dt):
    tend = s.cal_tend()
    s.step(dt, 3)
    return tend, s.get_field(dgk.FIELD_Q)


@pytest.mark.parametrize("form,p", [("HIP", p) for p in (1, 2, 4, 5, 7, 8, 11, 13, 15, 17)] +
                         [("HIP_MP", p) for p in (1, 2, 3, 4, 5, 6, 7, 9, 12, 15, 18)])
def test_constant_fields_equal_field_reads(monkeypatch, form, p):
    ne = (3, 2, 5) if p <= 7 else (2, 1, 3)
    q, u, v, w = inputs.random_fields(*ne, p, seed=800 + p, vel_scale=0.6)
    const = [np.full_like(q, c) for c in VEL]
    late = const[2].copy()
    late[-1, -1] *= 1.5  # one node differs, the last
    dt = 0.2 * inputs.cfl_dt(inputs.lgl_nodes(p), ne, (0.8, 0.8, 0.8))
    got = {}
    for env in ("1", "0"):
        monkeypatch.setenv("DGK_CVEL", env)
        with dgk.Solver.structured(form, *ne, p) as s:
            s.set_fields(q, *const)
            a = results(s, dt)
            s.set_fields(q, u, const[1], const[2])  # one component varies: the fields again
            b = results(s, dt)
            s.set_fields(q, const[0], const[1], late)
            c = results(s, dt)
            s.set_fields(q, *(2.0 * x for x in const))  # other constants
            d = results(s, dt)
            got[env] = a + b + c + d
    for k, (x, y) in enumerate(zip(got["1"], got["0"])):
        assert np.array_equal(x, y), k


def test_constant_wind_with_records_per_element(monkeypatch):
    """Several geometry records, each given the wind."""
    m = oracle.Mesh(3, 2, 2, 4)
    scale = 1.0 + 0.25 * np.arange(m.Ne)
    m.Escale = np.ascontiguousarray(m.Escale * scale[None, :, None])
    m.Fscale = np.ascontiguousarray(m.Fscale * scale[:, None])
    q = inputs.random_fields(3, 2, 2, 4, seed=12)[0]
    got = []
    for env in ("1", "0"):
        monkeypatch.setenv("DGK_CVEL", env)
        with dgk.Solver.create("HIP", m.Nq, m.Ne, m.NeA, m.NhaloNode, m.D, m.Lift, m.VMapM,
                               m.VMapP, m.halo_src_map, m.normal_fn, m.Escale, m.Fscale) as s:
            s.set_fields(q, *(np.full_like(q, c) for c in VEL))
            got.append(results(s, 1e-3))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
