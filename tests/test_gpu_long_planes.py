"""Planes with a row or column too long for the pencils (needs an MI355X): the
persistent kernels, with U3 and the scalars on the branch stream.

What this path alone has: COURANT's minimum taken by two streams and its
DELTA_T after they join, z transforms of more than 512 points, and more
(plane, field) items than scratch slots (256) in the transforms and in the
nonlinear pass.  RK3 steps of the deck with every term, DELTA_T variable,
against the oracle from the same state, each field within max(1e-11 per step,
4 x floor), the floor being what the oracle's own result changes under a 1e-16
perturbation of its input velocity; DELTA_T and TIME to 1e-12.  A row, column
or plane in the wrong place is O(1e-2) of the step's change."""
import pytest

from diablo_amd import channel, configs
from tests import helpers

pytestmark = pytest.mark.gpu

STATE = ("cu1", "cu2", "cu3", "cp")


def _oracle(dor, nx, ny, nz, n_th):
    p, gy, ic = configs.small_case(nx=nx, ny=ny, nz=nz, n_th=n_th)
    p.update(variable_dt=1, update_dt=1, cfl=0.3)
    o = dor.Oracle(p)
    o.set_grid_gy(gy)
    if n_th > 0:
        o.create_th(ic["th_ic_type"])
    o.create_flow(ic["ic_type"], ic["seed"], ic["amp"], ic["ymask"], ic["ubulk0"])
    return o, p, gy


@pytest.mark.parametrize("nx,ny,nz,n_th,steps", [(768, 6, 32, 1, 2), (32, 6, 768, 1, 2), (768, 136, 32, 0, 1)])
def test_long_plane_steps(oracle_mod, nx, ny, nz, n_th, steps):
    print(f"[long planes] {nx}x{ny}x{nz} n_th={n_th}, {steps} steps", flush=True)
    dor = oracle_mod
    o, p, gy = _oracle(dor, nx, ny, nz, n_th)
    o2, *_ = _oracle(dor, nx, ny, nz, n_th)
    helpers.perturb(dor, o2, 1e-16)
    ch = channel.Channel(p, gy)
    ch.upload(helpers.oracle_state(dor, o))
    ch.set_clock(0.0, p["delta_t"], 0)
    for q in (o, o2):
        q.time_step(steps)
    print("  oracle done", flush=True)
    ch.time_step(steps)
    t_o, dt_o, ts_o = o.clock()
    t_g, dt_g, _, ts_g = ch.clock()
    st = ch.download()
    ch.close()
    assert dt_o != p["delta_t"]  # COURANT has set it
    assert ts_g == ts_o == steps
    assert abs(dt_g - dt_o) <= 1e-12 * dt_o and abs(t_g - t_o) <= 1e-12 * t_o
    errs = helpers.field_errors(dor, o, st, keys=STATE)
    floor = helpers.field_errors(dor, o, helpers.oracle_state(dor, o2), keys=STATE)
    bad = helpers.within(errs, floor, 1e-11 * steps)
    assert not bad, (bad, errs, floor)
