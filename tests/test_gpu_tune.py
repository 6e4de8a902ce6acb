"""The autotuner: the shape it keeps is a pair that is fast together, and its
scratch trials leave the networks as they were; and a layout that it has to find."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_kept_shape_is_fast_in_a_trial():
    """Blocks of 64 for the integration and of 128 for the delivery are each
    among the fastest beside the other's default and 20 % slower together (20 000
    + 5 500 neurons); the kept shape's growth trial is held against the best of
    four plain pairs, with half of that as the margin."""
    from unsupervised_growth_amd import configs
    from unsupervised_growth_amd.engine import Engine
    net, kw = configs.c3()
    with Engine(ra_model=1, precision=1, **kw) as eng:
        eng.upload(net)

        def trial_ms(shape):
            eng.set_tuning(**shape)
            took = []
            for k in range(4):
                t0 = time.perf_counter()
                eng.run_trial(mode=0, training=True, trial_index=k, first_trial=k == 0, mean_injection_time=100.0)
                took.append(time.perf_counter() - t0)
            return 1000.0 * min(took)

        kept, _ = eng.autotune(windows=400)
        plain = [dict(kept, integrate_block=i, i_lanes=3, ra_lanes=0, deliver_block=d)
                 for i in (64, 256) for d in (64, 256)]
        took, best = trial_ms(kept), min(map(trial_ms, plain))
        print("kept", kept, "%.1f ms, best plain pair %.1f ms" % (took, best), flush=True)
        assert took < 1.1 * best


@pytest.mark.parametrize("precision", [0, 1])
def test_scratch_trials_leave_the_network(precision):
    """Weights, flags and lists (saturated rows among them) and the next growth
    trials are those of an engine that was not tuned."""
    from unsupervised_growth_amd.engine import Engine
    from unsupervised_growth_amd.network import random_network
    net = random_network(120, 40, n_train=12, p_ra2i=0.4, p_i2ra=0.2, seed=9)
    runs = []
    for tune in (False, True):
        with Engine(ra_model=1, precision=precision, trial_ms=120.0, seed=(4, 2)) as eng:
            eng.upload(net)
            out = [eng.run_trial(mode=0, training=True, trial_index=0, first_trial=True, mean_injection_time=20.0)]
            before = eng.download_synapses()
            if tune:
                shape = eng.tuning()
                eng.autotune(windows=200)
                eng.set_tuning(**shape)   # (in FP32 the rounding follows the layout)
            syn = [before, eng.download_synapses()]
            out.append(eng.run_trial(mode=0, training=True, trial_index=1, mean_injection_time=20.0))
            runs.append((out, syn + [eng.download_synapses()]))
    for s in (runs[1][1][0], runs[1][1][1]):
        for f in ("w", "act_cnt", "act_ids", "sup_cnt", "sup_ids", "remodeled"):
            np.testing.assert_array_equal(getattr(s, f), getattr(runs[0][1][0], f), err_msg=f)
    for f in ("w", "act_cnt", "act_ids", "sup_cnt", "sup_ids", "remodeled"):
        np.testing.assert_array_equal(getattr(runs[1][1][2], f), getattr(runs[0][1][2], f), err_msg=f)
    for a, b in zip(runs[0][0], runs[1][0]):
        for kind in ("soma", "dend", "interneuron"):
            for x, y in zip(getattr(a, kind), getattr(b, kind)):
                np.testing.assert_array_equal(x, y)
    assert sum(map(len, runs[0][0][1].soma)) > 0


def test_pool_is_tuned_on_chain_tests():
    """A serving pool's scratch trials are chain tests; its networks' results are
    those of a pool that was not tuned."""
    from unsupervised_growth_amd.configs import grown_chain_network
    from unsupervised_growth_amd.engine import Pool, pool_caps
    nets = [grown_chain_network(np.random.default_rng(k), 120 + 40 * k, 33 + 11 * k) for k in range(2)]
    caps = pool_caps(max_nets=2, max_ra=400, max_i=120, max_rr=4000, max_ra2i=20000, max_i2ra=20000,
                     max_in_degree=200, spikes_per_neuron=128)
    runs = []
    for tune in (False, True):
        with Pool(caps, ra_model=1, precision=0, trial_ms=100.0) as pool:
            handles = [pool.admit(net, (7 + k, 0)) for k, net in enumerate(nets)]
            if tune:
                _, ms = pool.autotune(windows=100)
                assert (ms > 0).all()
            trial = dict(mode=1, training=True, trial_index=0, first_trial=True, mean_injection_time=20.0)
            res = pool.run({h: trial for h in handles})
            runs.append([res[h] for h in handles])
    for a, b in zip(*runs):
        for kind in ("soma", "dend", "interneuron"):
            for x, y in zip(getattr(a, kind), getattr(b, kind)):
                np.testing.assert_array_equal(x, y)
        assert sum(map(len, a.soma)) > 0


def test_fp64_rk4_has_a_layout_between_octets_and_one_thread():
    """At 20 000 HVC-RA neurons four lanes per neuron take 61 us per window of
    k_integrate where eight take 76 and one thread 79."""
    from unsupervised_growth_amd import configs
    from unsupervised_growth_amd.engine import Engine
    net, kw = configs.c3()
    us = {}
    with Engine(ra_model=1, precision=0, **dict(kw, trial_ms=40.0)) as eng:
        eng.upload(net)
        eng.set_timing(True)
        for lanes in (1, 0):
            eng.set_tuning(ra_lanes=lanes)
            took = []
            for k in range(3):
                eng.set_timing(True)
                eng.run_trial(mode=0, training=True, trial_index=k, first_trial=k == 0, mean_injection_time=10.0)
                took.append(1000.0 * eng.kernel_timing("integrate")[0])
            us[lanes] = min(took)
    print("k_integrate us per window", us, flush=True)
    assert us[1] < 0.9 * us[0]
