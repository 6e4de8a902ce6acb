"""The decay at a growth trial's end, one wave per row, bit for bit against the
oracle: rows of 0 to 131 edges, weights on both sides of the thresholds and
flags that disagree with them, so every transition is met, several to a row."""
import numpy as np
import pytest

from oracle_lib import OracleSim
from test_oracle_pins import _net

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("degs", [(0, 1, 2), (63, 64, 65), (127, 128, 131)])
def test_row_transitions(degs):
    from unsupervised_growth_amd.engine import Engine
    from unsupervised_growth_amd.network import NoiseParams, SynapticParams
    rng = np.random.default_rng(degs[0])
    n, syn = 140, SynapticParams()
    thr = [0.0, syn.BETA, syn.ACTIVATION_THRESHOLD, syn.SUPERSYNAPSE_THRESHOLD]
    rr, active, supers = [], [], []
    for i in range(n):
        tg = np.sort(rng.choice([j for j in range(n) if j != i], degs[i % 3], replace=False))
        w = rng.choice(thr, len(tg)) + rng.choice([0.0, 0.5, 1.5, -0.5], len(tg)) * syn.BETA
        rr += [(i, int(j), 1.0, float(max(x, 0.0))) for j, x in zip(tg, w)]
        active += [(i, int(j)) for j in tg if rng.random() < 0.5]
        supers += [(i, int(j)) for j in rng.permutation(tg)[:rng.integers(0, syn.Nss + 1)]]
    net = _net(n, 0, rr=rr, active=active, supers=supers, remodeled=rng.integers(0, 2, n))
    kw = dict(trial_ms=1.0, i_poisson=0, noise=NoiseParams(0.0, 0.0, 0.0, 0.0), syn=syn)
    ora = OracleSim(net, **kw)
    with Engine(**kw) as eng:
        eng.upload(net)
        for k in range(3):
            tr = dict(mode=0, training=False, trial_index=k, first_trial=k == 0, mean_injection_time=100.0)
            o, r = ora.run_trial(**tr), eng.run_trial(**tr)
            assert r.warnings == o["warnings"]
            s, want = eng.download_synapses(), ora.synapses()
            for f in ("w", "act_cnt", "act_ids", "sup_cnt", "sup_ids", "remodeled"):
                np.testing.assert_array_equal(getattr(s, f), want[f], err_msg=f)
