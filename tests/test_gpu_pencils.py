"""Large planes as pencils, and the persistent kernels beyond them (needs an
MI355X): x lengths whose row blocks leave threads over and whose last row
block and last column tile are partly empty, scalars with both wall types,
a grid whose planes take the scratch in two parts, and a row too long for the
pencils.

One RK3 step of the deck with every term against the oracle from the same
state, each field within max(1e-11, 4 x floor), the floor being what the
oracle's own result changes under a 1e-16 perturbation of its input velocity.
A row, column or product in the wrong place is O(1e-2) of the step's change.
"""
import pytest

from diablo_amd import channel
from tests import helpers

pytestmark = pytest.mark.gpu

STATE = ("cu1", "cu2", "cu3", "cp")


@pytest.mark.parametrize("nx,ny,nz,n_th", [
    (192, 9, 144, 2), (324, 6, 96, 0), (256, 64, 256, 4), (768, 6, 32, 1)])
def test_large_plane_step(oracle_mod, nx, ny, nz, n_th):
    print(f"[pencils] {nx}x{ny}x{nz} n_th={n_th}", flush=True)
    dor = oracle_mod
    kw = dict(nx=nx, ny=ny, nz=nz, n_th=n_th)
    o, p, gy, ic = helpers.make_oracle(dor, "small_case", **kw)
    o2, *_ = helpers.make_oracle(dor, "small_case", **kw)
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
