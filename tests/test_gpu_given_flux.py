"""dgk_cal_dqdt from a given face flux: the staged and the register form give the
same bits (launch-wide and per-element geometry, tilted normals, a constant wind,
partial workgroups), and the register form, which the defaults take at p = 4 and
6..13, is the faster one there."""
import numpy as np
import pytest

import dgk
import oracle
from dgk import inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mesh", ["box", "records", "tilted", "constant"])
@pytest.mark.parametrize("p", [1, 2, 3, 4, 6, 7, 8, 11, 13, 15])
def test_forms_agree(p, mesh):
    ne = (3, 2, 3) if p <= 7 else (2, 1, 2)
    m = oracle.Mesh(*ne, p)
    if mesh == "records":
        scale = 1.0 + 0.25 * np.arange(m.Ne)
        m.Escale = np.ascontiguousarray(m.Escale * scale[None, :, None])
        m.Fscale = np.ascontiguousarray(m.Fscale * scale[:, None])
    elif mesh == "tilted":
        m.normal_fn = np.ascontiguousarray(m.normal_fn + 0.05)
    q, u, v, w = inputs.random_fields(*ne, p, seed=70 + p, vel_scale=0.7)
    if mesh == "constant":
        u, v, w = (np.full_like(q, c) for c in (0.4, -0.3, 0.55))
    flux = np.random.RandomState(p).uniform(-1.0, 1.0, (m.Ne, m.NfpTot))
    ref = m.cal_dqdt(m.field(q), m.field(u), m.field(v), m.field(w), flux)
    got = []
    try:
        for cand in (-1, 0, 1):
            dgk.tile_select("HIP", p, cand)
            with dgk.Solver.create("HIP", m.Nq, m.Ne, m.NeA, m.NhaloNode, m.D, m.Lift, m.VMapM,
                                   m.VMapP, m.halo_src_map, m.normal_fn, m.Escale, m.Fscale) as s:
                s.set_fields(q, u, v, w)
                s.cal_dqdt(flux)
                got.append(s.get_field(dgk.FIELD_DQDT))
    finally:
        dgk.tile_select("HIP", p, -1)
    assert np.array_equal(got[1], got[0]) and np.array_equal(got[2], got[0])
    assert np.abs(got[0] - ref).max() <= 1e-13 * np.abs(ref).max()


@pytest.mark.parametrize("p,ne", [(7, 32), (13, 18)])
def test_default_is_the_register_form(p, ne):
    """Measured: 140 against 182 us at p = 7, 171 against 292 at p = 13."""
    def per_launch(s):
        for _ in range(10):
            s.cal_dqdt()
        s.synchronize()
        s.timer_reset()
        s.set_kernel_timing(True)
        for _ in range(30):
            s.cal_dqdt()
        s.synchronize()
        s.set_kernel_timing(False)
        seconds, n = s.timers()["Volume derivate + surface lift"]
        return seconds / n

    with dgk.Solver.structured("HIP", ne, ne, ne, p) as s:
        s.init_gaussian((0.3, 0.4, 0.5), 0.1, (0.3, -0.7, 0.5))
        s.cal_elembnd_flux(download=False)
        default = min(per_launch(s) for _ in range(3))
        try:
            dgk.tile_select("HIP", p, 0)
            staged = min(per_launch(s) for _ in range(3))
        finally:
            dgk.tile_select("HIP", p, -1)
    assert default < 0.9 * staged, (default, staged)
