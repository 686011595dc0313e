"""Rounding of the FP64 column solve (needs an MI355X): every row of every
segment is the reference's own operation on its neighbour (mpi.f:630-703,
767-809), only the values carried into a segment are composed.

Velocities that depend on y alone, random in every row, and a viscous number
of about 1e-8: then nothing but the solve rounds (the transforms of a constant
plane are exact, the explicit half is far below its row's last digit), and a
carry is its end row's value to the last bit, as what it hands on from further
away is below 1e-30 of it.  So a substep must give the oracle's one sweep bit
for bit; a row that gets its carry as a term added afterwards does not (one
more rounding)."""
import numpy as np
import pytest

from diablo_amd import channel, configs
from tests import helpers

pytestmark = pytest.mark.gpu


def _substep(dor, ny, bc):
    p = configs.base_params(8, ny, 4)
    dy = 2.0 / ny
    p.update(nu=4e-5 * dy * dy, u_bc_ymin=bc, u_bc_ymax=bc, w_bc_ymin=bc, w_bc_ymax=bc, u_bc_ymin_c1=0.5 * (1 - bc),
             w_bc_ymax_c1=-0.25 * (1 - bc))
    gy = configs.make_gy(ny, 2.0, 0.0, 2)
    o = dor.Oracle(p)
    o.set_grid_gy(gy)
    rng = np.random.default_rng(ny)
    for w in (dor.CU1, dor.CU3):
        o.carr(w)[:, 0, 0] = rng.standard_normal(ny + 2)
    ch = channel.Channel(p, gy)
    ch.upload(helpers.oracle_state(dor, o))
    ch.set_clock(0.0, p["delta_t"], 0)
    o.rk_chan_1(1)
    ch.rk_substep(1)
    st = ch.download()
    ch.close()
    for k, w in (("cu1", dor.CU1), ("cu3", dor.CU3)):
        got, ref = st[k][:, 0, 0], o.carr(w)[:, 0, 0]
        off = np.flatnonzero(got != ref)
        assert off.size == 0, (k, off, np.abs(got - ref).max())


@pytest.mark.parametrize("ny", [65, 129, 193, 257])  # 5, 9, 13 and 17 rows per segment
def test_rows_are_the_sweeps_own(oracle_mod, ny):
    print(f"[solve rows] ny={ny}", flush=True)
    _substep(oracle_mod, ny, 0)


@pytest.mark.parametrize("ny", [40, 65, 127, 129, 192, 257])
def test_pivots_are_the_recurrence_own(oracle_mod, ny):
    """Free-slip walls: the wall row's multiplier is 1/pivot of the row below
    it, so the pivot that a lane of the tables' scan starts from shows in the
    wall value; at NY = 129 and 192 the row is a lane's first."""
    print(f"[solve rows] free-slip ny={ny}", flush=True)
    _substep(oracle_mod, ny, 1)
