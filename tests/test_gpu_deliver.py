"""Chain-test RA->RA pushes (four lanes per neuron when no network grows), bit
for bit against the oracle: rows of 0 to 9 active edges, delays of none, of
exact steps and of several windows, windows of 1 to 63 steps (the arrival
step's search)."""
import numpy as np
import pytest

from oracle_lib import OracleSim
from test_oracle_pins import DT, _net

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lists", [1, 0])
@pytest.mark.parametrize("sync_ms", [0.02, 0.25, 1.25])
def test_chain_push_lanes(lists, sync_ms):
    from unsupervised_growth_amd.engine import Engine
    delays = [0.0, DT, 2 * DT, 0.25, 0.2500001, 0.37, 1.0, 3.3, 5.0]
    rr = [(i, j, delays[(i + j) % 9], 8.0) for i in range(10) for j in range(12) if j != i]
    active = [(i, (i + 1 + k) % 12) for i in range(10) for k in range(i)]
    net = _net(12, 0, rr=rr, active=active, train=[3, 9], spread=[0.0, 2.0])
    kw = dict(trial_ms=40.0, sync_ms=sync_ms)
    ora = OracleSim(net, **kw)
    fired = 0
    with Engine(**kw) as eng:
        eng.upload(net)
        eng.set_tuning(deliver_lists=lists, deliver_block=64)
        for k in range(2):
            tr = dict(mode=1, trial_index=k, mean_injection_time=10.0)
            o, r = ora.run_trial(**tr), eng.run_trial(want_state=True, **tr)
            for kind in ("soma", "dend"):
                for a, b in zip(getattr(r, kind), o[kind]):
                    np.testing.assert_array_equal(a, b)
            np.testing.assert_array_equal(r.ra_state, o["ra_state"])
            fired += sum(map(len, r.soma))
    assert fired > 4
