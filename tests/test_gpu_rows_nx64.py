"""The nonlinear pass with x rows of NX = 64 in registers (needs an MI355X): one to
four slabs of 16 rows, with none to two scalars, and with the LES model.

Three RK substeps of the deck with every term (rotation, forcing, buoyancy,
mixed walls) against the oracle from the same state, each field within
max(1e-11, 4 x floor), the floor being what the oracle's own result changes
under a 1e-16 perturbation of its input velocity.  A sample or a product in the
wrong place is O(1e-2) of a substep's change."""
import pytest

from diablo_amd import channel
from tests import helpers

pytestmark = pytest.mark.gpu

STATE = ("cu1", "cu2", "cu3", "cp")


@pytest.mark.parametrize("name,nz,n_th", [("small_case", 16, 1), ("small_case", 48, 0), ("small_case", 64, 2),
                                          ("les_small", 32, 1), ("les_small", 64, 0)])
def test_substeps_with_rows_in_registers(oracle_mod, name, nz, n_th):
    print(f"[rows nx64] {name} 64x9x{nz} n_th={n_th}", flush=True)
    dor = oracle_mod
    kw = dict(nx=64, ny=9, nz=nz, n_th=n_th)
    o, p, gy, ic = helpers.make_oracle(dor, name, **kw)
    o2, *_ = helpers.make_oracle(dor, name, **kw)
    helpers.perturb(dor, o2, 1e-16)
    ch = channel.Channel(p, gy)
    ch.upload(helpers.oracle_state(dor, o))
    ch.set_clock(0.0, p["delta_t"], 0)
    for q in (o, o2):
        q.time_step(1)
    ch.time_step(1)
    st = ch.download()
    errs = helpers.field_errors(dor, o, st, keys=STATE)
    floor = helpers.field_errors(dor, o, helpers.oracle_state(dor, o2), keys=STATE)
    ch.close()
    bad = helpers.within(errs, floor, 1e-11)
    assert not bad, (bad, errs, floor)
