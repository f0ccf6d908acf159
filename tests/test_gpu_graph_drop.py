"""Settings that drop the captured cycle while replays of it are queued: the replays finish first,
and the run goes on as if it had been waited for."""
import numpy as np
import pytest

from parthenon_amd import _check, lib
from parthenon_amd.burgers import DeviceBurgersDriver, make_burgers_mesh

pytestmark = pytest.mark.gpu

DROPS = {
    "time-limits": lambda d: d.set_time_limits(tlim=1e9),
    "tuning": lambda d: d.set_tuning(d.tuning()),
    "split": lambda d: _check(lib().pth_burgers_set_sweep_split(d.mesh._h, 1), "split"),
    "stage-form": lambda d: _check(lib().pth_burgers_set_sweep(d.mesh._h, 1), "sweep"),
}


@pytest.mark.parametrize("name", list(DROPS))
def test_queued_replays_finish(name):
    print(f"case graph drop {name}", flush=True)
    got = []
    for wait in (False, True):
        d = DeviceBurgersDriver(make_burgers_mesh((32, 32, 32), (16, 16, 16), 4, 2), sweep=True)
        d.initialize("sinusoid", seed=4)
        d.cycles(40)
        if wait:
            d.synchronize()
        DROPS[name](d)
        d.cycles(2)
        got.append((d.base.download("U"), d.clock()))
    assert got[0][1] == got[1][1] and np.array_equal(got[0][0], got[1][0])
