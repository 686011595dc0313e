"""The Crank-Nicolson tables rebuilt for COURANT's DELTA_T (needs an MI355X):
their pivots come from a scan over a wave's lanes, one to five rows a lane.
The fewest rows, one row more than the lanes hold with one, two and four rows
each, and the most; ordinary viscosity and rows a hundred times as stiff, where
the pivots below a wall gradient are most sensitive.  (Two scalars, so that
both kinds of wall appear on both sides.)

Two steps with DELTA_T from the CFL condition against the oracle from the same
state, each field within max(1e-11, 4 x floor), the floor being what the
oracle's own result changes under a 1e-16 perturbation of its input velocity,
and the clock to 1e-11.  A pivot from a wrong row is O(1e-2) of a step's
change."""
import numpy as np
import pytest

from diablo_amd import channel, configs
from tests import helpers

pytestmark = pytest.mark.gpu

STATE = ("cu1", "cu2", "cu3")


@pytest.mark.parametrize("ny,nu", [(4, 0.01), (62, 0.01), (63, 1.0), (127, 0.01), (127, 1.0), (255, 1.0), (286, 0.01)])
def test_tables_of_a_new_time_step(oracle_mod, ny, nu):
    print(f"[cn pivots] NY={ny} nu={nu}", flush=True)
    dor = oracle_mod

    def start():
        p, gy, ic = configs.small_case(8, ny, 4, 2)
        p.update(nu=nu, variable_dt=1, cfl=0.3, update_dt=1)
        o = dor.Oracle(p)
        o.set_grid_gy(gy)
        o.create_th(ic["th_ic_type"])
        o.create_flow(ic["ic_type"], ic["seed"], ic["amp"], ic["ymask"], ic["ubulk0"])
        return o, p, gy

    (o, p, gy), (o2, _, _) = start(), start()
    helpers.perturb(dor, o2, 1e-16)
    ch = channel.Channel(p, gy)
    ch.upload(helpers.oracle_state(dor, o))
    ch.set_clock(0.0, p["delta_t"], 0)
    for q in (o, o2):
        q.time_step(2)
    ch.time_step(2)
    st = ch.download()
    errs = helpers.field_errors(dor, o, st, keys=STATE)
    floor = helpers.field_errors(dor, o, helpers.oracle_state(dor, o2), keys=STATE)
    time, dt, _, step = ch.clock()
    ch.close()
    want = o.clock()
    assert step == want[2] == 2 and dt != p["delta_t"]
    np.testing.assert_allclose([time, dt], want[:2], rtol=1e-11)
    bad = helpers.within(errs, floor, 1e-11)
    assert not bad, (bad, errs, floor)
