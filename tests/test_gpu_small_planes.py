"""The nonlinear pass of small planes (needs an MI355X): fewer complex values
than a block has threads, two samples and two modes per thread with a
remainder, tall and wide planes, the largest plane of the small path and the
next one beyond it, with none to four scalars, and with the LES model.

Three RK substeps of the deck with every term (rotation, forcing, buoyancy,
mixed walls) against the oracle from the same state, each field within
max(1e-11, 4 x floor), the floor being what the oracle's own result changes
under a 1e-16 perturbation of its input velocity.  A sample, mode or product
in the wrong place is O(1e-2) of a substep's change."""
import numpy as np
import pytest

from diablo_amd import channel
from tests import helpers

pytestmark = pytest.mark.gpu

STATE = ("cu1", "cu2", "cu3", "cp")


@pytest.mark.parametrize("name,nx,nz,n_th", [
    ("small_case", 8, 4, 1), ("small_case", 256, 4, 1), ("small_case", 24, 64, 0), ("small_case", 96, 6, 4),
    ("small_case", 48, 36, 2), ("small_case", 256, 8, 1), ("les_small", 48, 32, 1)])
def test_small_plane_substeps(oracle_mod, name, nx, nz, n_th):
    print(f"[small planes] {name} {nx}x9x{nz} n_th={n_th}", flush=True)
    dor = oracle_mod
    kw = dict(nx=nx, ny=9, nz=nz, n_th=n_th)
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
