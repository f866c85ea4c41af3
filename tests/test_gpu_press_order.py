"""The step's two routes from the advanced velocity to the filtered state: the
pressure's right-hand side formed inside its row transform, in FP64 with the
filter in front of the projection (plain steps), and the prepared right-hand
side with the filter behind (statistics steps, which sample the unfiltered
velocity).  LES_FUSE=0 keeps the first route (its filter as a pass of its
own), so the comparison with it does not see the order.

Both are held to the oracle elsewhere, at TOL in FP64 and MIX_STATE in the
mixed mode, so they may differ by twice that.  dp/dz is formed in the
projection from the p that is stored, rounded as it is stored: to the bit."""
import numpy as np
import pytest

from overlappingbls_amd import config
from overlappingbls_amd.abi import LES_MIXED

from test_gpu_mixed import MIX_STATE
from test_gpu_parity import TOL, rel

pytestmark = pytest.mark.gpu


# land_lbc0: the surface-temperature term of the bottom row; mid_rect, wide:
# sides of different plans; ocean: a stress-free and a wall boundary
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("case", ["small", "mid", "mid_rect", "wide", "land_lbc0", "land_damp2", "ocean_sbl"])
def test_press_routes_agree(case, mixed, gpu_lib):
    nl = config.workload(case)
    p = nl.params()
    f = config.initial_fields(nl, seed=61, vw_noise=True)
    ctx = []
    for stats in (False, True):
        g = gpu_lib.create(p)
        if mixed:
            g.set_precision(LES_MIXED)
        if stats:
            g.set_avgslice(True, 1, 1000)
        config.load_state(g, f)
        ctx.append(g)
    a, b = ctx
    bound = 2.0 * (MIX_STATE if mixed else TOL)
    dz = p.lz_tot / (p.nzt - 1)
    for jt in (1, 2, 3):
        for g in ctx:
            g.run(jt, 1)
        bad = {}
        for n in ("U", "V", "W", "THETA"):
            sl = config.physical_levels(n, p.nzt)
            r = rel(a.get(n)[sl], b.get(n)[sl])
            if not r <= bound:
                bad[n] = r
        assert not bad, (jt, bad)
        for g in ctx:
            pr, pz = g.get("P"), g.get("DPDZ")[1:p.nzt]
            d = (pr[1:p.nzt] - pr[:p.nzt - 1]) / dz
            assert np.array_equal(pz, d.astype(np.float32).astype(np.float64) if mixed else d)
    # the routes do differ
    assert any(not np.array_equal(a.get(n), b.get(n)) for n in ("U", "V", "W"))
