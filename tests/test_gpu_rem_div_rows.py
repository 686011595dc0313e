"""REM_DIV_CHAN at the edges of its split of a mode's rows over threads (needs
an MI355X): the fewest rows, one row more than a wave's groups and than a
block's groups hold with one row each, the last NY with 32 threads per mode
and the first with 64, an uneven last group, and the most rows.

Against the oracle's projection of the same random field, each field within
max(1e-11, 4 x floor), the floor being what the oracle's own result changes
under a 1e-16 perturbation of its input (the sweeps' rounding is amplified by
the Poisson matrix).  A lost carry between threads or waves is O(1)."""
import numpy as np
import pytest

from diablo_amd import channel
from tests import helpers

pytestmark = pytest.mark.gpu

STATE = ("cu1", "cu2", "cu3")


@pytest.mark.parametrize("ny", [4, 10, 34, 66, 161, 162, 250, 286])
def test_rem_div_at_row_group_edges(oracle_mod, ny):
    print(f"[rem_div] NY={ny}", flush=True)
    dor = oracle_mod

    def noisy():
        o, p, gy, ic = helpers.make_oracle(dor, "small_case", ny=ny)
        rng = np.random.default_rng(3)
        for w in (dor.CU1, dor.CU2, dor.CU3):
            blk = o.carr(w)[:, : o.tnkz + 1, : o.nkx + 1]
            blk += 0.01 * (rng.standard_normal(blk.shape) + 1j * rng.standard_normal(blk.shape))
        return o, p, gy

    (o, p, gy), (o2, _, _) = noisy(), noisy()
    helpers.perturb(dor, o2, 1e-16)
    ch = channel.Channel(p, gy)
    ch.upload(helpers.oracle_state(dor, o))
    for q in (o, o2):
        q.rem_div()
    ch.rem_div()
    st = ch.download()
    errs = helpers.field_errors(dor, o, st, keys=STATE)
    floor = helpers.field_errors(dor, o, helpers.oracle_state(dor, o2), keys=STATE)
    ch.close()
    bad = helpers.within({k: errs[k] for k in STATE}, floor, 1e-11)
    assert not bad, (bad, errs, floor)
