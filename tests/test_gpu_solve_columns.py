"""The FP64 column solve at the edges of its split (needs an MI355X): the
fewest rows (segments of one row, most of them empty), the last and the first
NY+2 of each row count per thread, the most rows, and planes of 32, 48 and 72
columns (blocks take 32).  And a context switched to the mixed form and back,
whose tables are laid out anew each time.

Two steps with two scalars, mixed walls and DELTA_T from the CFL condition
(whose minimum the solve finds) against the oracle from the same state, each
field within max(1e-11, 4 x floor), the floor being what the oracle's own
result changes under a 1e-16 perturbation of its input velocity.  A lost carry
or a row of another segment is O(1e-2) of a step's change."""
import numpy as np
import pytest

from diablo_amd import channel, configs
from tests import helpers

pytestmark = pytest.mark.gpu

STATE = ("cu1", "cu2", "cu3")


def start(dor, nx, ny, nz):
    p, gy, ic = configs.small_case(nx, ny, nz, 2)
    p.update(variable_dt=1, cfl=0.3, update_dt=1)
    o = dor.Oracle(p)
    o.set_grid_gy(gy)
    o.create_th(ic["th_ic_type"])
    o.create_flow(ic["ic_type"], ic["seed"], ic["amp"], ic["ymask"], ic["ubulk0"])
    return o, p, gy


@pytest.mark.parametrize("nx,ny,nz", [(8, 4, 4), (8, 78, 6), (12, 79, 4), (8, 142, 4), (12, 143, 6), (8, 206, 6),
                                      (12, 207, 4), (8, 286, 4)])
def test_column_solve_edges(oracle_mod, nx, ny, nz):
    print(f"[solve columns] {nx}x{ny}x{nz}", flush=True)
    dor = oracle_mod
    (o, p, gy), (o2, _, _) = start(dor, nx, ny, nz), start(dor, nx, ny, nz)
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
    dt = ch.clock()[1]
    ch.close()
    np.testing.assert_allclose(dt, o.clock()[1], rtol=1e-11)
    bad = helpers.within(errs, floor, 1e-11)
    assert not bad, (bad, errs, floor)


def test_switching_forms_lays_the_tables_out_anew(oracle_mod):
    print("[solve columns] mixed and back", flush=True)
    dor = oracle_mod
    o, p, gy = start(dor, 16, 17, 8)
    p["variable_dt"] = 0  # the tables of the grid serve every step
    out = []
    for switch in (False, True):
        ch = channel.Channel(p, gy)
        ch.upload(helpers.oracle_state(dor, o))
        ch.set_clock(0.0, p["delta_t"], 0)
        if switch:
            ch.set_mixed_precision(True)
            ch.time_step(1)
            ch.set_mixed_precision(False)
            ch.upload(helpers.oracle_state(dor, o))
            ch.set_clock(0.0, p["delta_t"], 0)
        ch.time_step(2)
        out.append(ch.download())
        ch.close()
    for k in ("cu1", "cu2", "cu3", "cp", "cth"):
        assert np.array_equal(out[0][k], out[1][k]), k
