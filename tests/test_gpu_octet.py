"""The FP64 octet steppers (eight lanes per neuron) where they can go wrong, bit
for bit against the oracle: partly filled waves, steps that leave the range of
the fast quotients and repeat with IEEE division, and networks too large for
octets, which take four lanes or one thread per neuron."""
import dataclasses

import numpy as np
import pytest

from oracle_lib import OracleSim

pytestmark = pytest.mark.gpu


def _compare(net, trial_ms, trials=1, tuning=None, **kw):
    from unsupervised_growth_amd.engine import Engine
    ora = OracleSim(net, trial_ms=trial_ms, **kw)
    with Engine(trial_ms=trial_ms, **kw) as eng:
        eng.upload(net)
        if tuning:
            eng.set_tuning(**tuning)
        for k in range(trials):
            tr = dict(mode=0, trial_index=k, first_trial=k == 0, mean_injection_time=5.0)
            o, r = ora.run_trial(**tr), eng.run_trial(want_state=True, **tr)
            for kind in ("soma", "dend", "interneuron"):
                for a, b in zip(getattr(r, kind), o[kind]):
                    np.testing.assert_array_equal(a, b)
            np.testing.assert_array_equal(r.ra_state, o["ra_state"])
            np.testing.assert_array_equal(r.i_state, o["i_state"])
    return r


@pytest.mark.parametrize("model", [0, 1])
@pytest.mark.parametrize("n_ra,n_i", [(1, 1), (7, 9), (8, 8), (65, 17)])
def test_partly_filled_waves(model, n_ra, n_i):
    from unsupervised_growth_amd.network import random_network
    net = random_network(n_ra, n_i, n_train=4, p_ra2i=0.5, p_i2ra=0.5, seed=n_ra)
    _compare(net, 60.0, trials=2, ra_model=model, ra_poisson=model,
             tuning=dict(integrate_block=64 if n_ra < 60 else 256))


@pytest.mark.parametrize("model", [0, 1])
@pytest.mark.parametrize("sync_ms", [0.02, 0.35, 0.37, 1.25])
def test_window_tables(model, sync_ms):
    """Windows of 1 to 63 steps: the tables that a block of 64 stages with one
    round of loads (18 steps) and the ones that take more, in FP64 and, against
    blocks of 256, in FP32."""
    from unsupervised_growth_amd.engine import Engine
    from unsupervised_growth_amd.network import random_network
    net = random_network(20, 12, n_train=4, p_ra2i=0.5, p_i2ra=0.5, seed=5)
    kw = dict(ra_model=model, ra_poisson=model, sync_ms=sync_ms)
    _compare(net, 20.0, tuning=dict(integrate_block=64), **kw)
    states = []
    for block in (64, 256):
        with Engine(precision=1, trial_ms=20.0, **kw) as eng:
            eng.upload(net)
            eng.set_tuning(integrate_block=block)
            r = eng.run_trial(mode=0, trial_index=0, first_trial=True, mean_injection_time=5.0, want_state=True)
            states.append((r.ra_state, r.i_state))
    for a, b in zip(*states):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("model", [0, 1])
def test_steps_out_of_the_fast_range(model):
    """Resting potentials far out (gate arguments and voltages beyond the fast
    range, overflowing exponentials) and conductances under which the HVC-I
    stepper diverges through every magnitude to infinity and NaN."""
    from unsupervised_growth_amd.network import random_network
    net = random_network(24, 12, n_train=12, p_ra2i=0.6, p_i2ra=0.6, seed=2)
    erest = net.erest.copy()
    erest[:4] = [-3.0e4, 3.0e4, -1.0e9, 2.0e5]
    net = dataclasses.replace(net, erest=erest, ra2i_w=net.ra2i_w * 1.0e5)
    r = _compare(net, 30.0, ra_model=model)
    assert r.bad_values == -1 and not np.isfinite(r.i_state).all() and (abs(r.ra_state[:4, 0]) > 2000).any()


def _padded(small, n_ra):
    """The network with n_ra - small.n_ra unconnected HVC-RA neurons after its own."""
    pad = n_ra - small.n_ra

    def more(ptr):
        return np.concatenate([ptr, np.full(pad, ptr[-1], np.int32)])

    z = np.zeros(pad, np.int32)
    return dataclasses.replace(small, n_ra=n_ra, ra2i_ptr=more(small.ra2i_ptr), rr_ptr=more(small.rr_ptr),
                               act_cnt=np.concatenate([small.act_cnt, z]), sup_cnt=np.concatenate([small.sup_cnt, z]),
                               remodeled=np.concatenate([small.remodeled, z]),
                               erest=np.concatenate([small.erest, np.linspace(-90.0, -60.0, pad)]),
                               gca=np.concatenate([small.gca, np.linspace(0.0, 60.0, pad)]))


@pytest.mark.parametrize("model,n_ra", [(0, 32769), (1, 26625)])
def test_large_network_takes_one_thread_per_neuron(model, n_ra):
    from unsupervised_growth_amd.network import random_network
    small = random_network(5, 3, n_train=2, p_ra2i=0.5, p_i2ra=0.5, seed=4, rr=2)
    _compare(_padded(small, n_ra), 3.0, ra_model=model)


@pytest.mark.parametrize("model,n_ra,ra_lanes", [(1, 14337, 1), (0, 32769, 0), (1, 26625, 0)])
def test_large_network_through_a_kick(model, n_ra, ra_lanes):
    """The layouts of large networks (four lanes in the RK4 model, one thread)
    with their spikes, deliveries and STDP: two trials kicked at their start."""
    from unsupervised_growth_amd.engine import Engine
    from unsupervised_growth_amd.network import random_network
    small = random_network(20, 6, n_train=8, p_ra2i=0.5, p_i2ra=0.5, seed=4, w_rr=150.0, delays=("uniform", 0.0, 2.0),
                           rr_delays=("uniform", 0.0, 2.0))
    net = _padded(small, n_ra)
    kw = dict(ra_model=model, ra_poisson=model, trial_ms=9.0)
    ora = OracleSim(net, **kw)
    with Engine(**kw) as eng:
        eng.upload(net)
        eng.set_tuning(ra_lanes=ra_lanes)
        for k in range(2):
            tr = dict(mode=0, trial_index=k, first_trial=k == 0, mean_injection_time=0.5)
            o, r = ora.run_trial(**tr), eng.run_trial(want_state=True, **tr)
            for kind in ("soma", "dend", "interneuron"):
                for a, b in zip(getattr(r, kind), o[kind]):
                    np.testing.assert_array_equal(a, b)
            np.testing.assert_array_equal(r.ra_state, o["ra_state"])
            np.testing.assert_array_equal(r.i_state, o["i_state"])
            s, want = eng.download_synapses(), ora.synapses()
            for f in ("w", "act_cnt", "act_ids", "sup_cnt", "sup_ids", "remodeled"):
                np.testing.assert_array_equal(getattr(s, f), want[f], err_msg=f)
            for kind in ("soma", "dend", "interneuron"):
                assert sum(map(len, getattr(r, kind)[:20])) > 0, kind
            assert (s.w != small.rr_w).all() and s.act_cnt.any()
            # inhibition and, once synapses are active, excitation has reached the neurons
            assert (r.ra_state[:20, 11] > 0).any() and (r.i_state[:, 5] > 0).any()


@pytest.mark.parametrize("model,poisson", [(0, 0), (1, 1)])
@pytest.mark.parametrize("n,steps", [(1, 1), (8, 32), (9, 33), (33000, 3)])
def test_trace_ra_sizes(model, poisson, n, steps):
    """Chunk and block edges; the last size is beyond the octets."""
    from oracle_lib import oracle, ra_inputs, run_ra_trace
    from unsupervised_growth_amd.engine import Engine
    inp = ra_inputs(n, steps, kick_step=min(2, steps - 1))
    ref_state, ref_fired = run_ra_trace(oracle(), "ora", model, inp, poisson=poisson, seed=(7, 0), trial=2)
    with Engine(ra_model=model, ra_poisson=poisson, seed=(7, 0)) as eng:
        st, fi = eng.trace_ra(*inp, trial=2)
    np.testing.assert_array_equal(fi, ref_fired)
    np.testing.assert_array_equal(st, ref_state)


@pytest.mark.parametrize("n,steps", [(1, 1), (8, 32), (9, 33), (24577, 14)])
def test_trace_i_sizes(n, steps):
    from oracle_lib import i_inputs, oracle, run_i_trace
    from unsupervised_growth_amd.engine import Engine
    inp = i_inputs(n, steps, exc_scale=0.3)
    ref_state, ref_fired = run_i_trace(oracle(), "ora", 0, inp, first_trial=0, seed=(7, 0), trial=3)
    with Engine(seed=(7, 0)) as eng:
        st, fi = eng.trace_i(*inp, trial=3)
    np.testing.assert_array_equal(fi, ref_fired)
    np.testing.assert_array_equal(st, ref_state)


@pytest.mark.parametrize("model,ra_lanes", [(1, 0), (1, 1), (0, 0)])
def test_fp32_one_thread_shape_on_octets(model, ra_lanes):
    """A small FP32 network whose shape asks for one thread per HVC-I neuron
    equals the same network in a batch too large for octets (spikes: the rates
    pass their series near v = -15 and v = -22)."""
    from unsupervised_growth_amd.engine import Engine
    from unsupervised_growth_amd.network import random_network
    net = random_network(40, 37, n_train=8, p_ra2i=0.5, p_i2ra=0.3, gei_max=2.0, seed=3)
    i = 10241
    z, f = np.zeros(2, np.int32), np.zeros(0, np.int32)
    e = np.zeros(0)
    idle = dataclasses.replace(net, n_ra=1, n_i=i, ra2i_ptr=z, ra2i_tgt=f, ra2i_w=e, ra2i_d=e,
                               i2ra_ptr=np.zeros(i + 1, np.int32), i2ra_tgt=f, i2ra_w=e, i2ra_d=e, rr_ptr=z, rr_tgt=f,
                               rr_d=e, rr_w=e, act_cnt=z[:1], act_ids=f, sup_cnt=z[:1], sup_ids=f, remodeled=z[:1],
                               erest=net.erest[:1], gca=net.gca[:1], train_ids=f, spread=e)
    kw = dict(precision=1, trial_ms=100.0, ra_model=model)
    tr = dict(mode=0, trial_index=0, first_trial=True, mean_injection_time=10.0)
    with Engine(seed=(5, 0), **kw) as a, Engine(**kw) as b:
        a.upload(net)
        b.upload_batch([net, idle], [(5, 0), (6, 0)])
        for x in (a, b):
            x.set_tuning(i_lanes=0, ra_lanes=ra_lanes)
        ra, rb = a.run_trial(**tr), b.run_batch([tr, tr])[0]
    assert sum(map(len, ra.interneuron)) > 0
    for kind in ("soma", "dend", "interneuron"):
        for x, y in zip(getattr(ra, kind), getattr(rb, kind)):
            np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("model,ra_lanes", [(1, 0), (1, 1), (0, 0)])
def test_fp32_one_thread_arithmetic_has_one_definition(model, ra_lanes):
    """The same, state by state and bit for bit: one network alone and with idle
    HVC-I neurons after its own, enough of them that the kernel takes one
    thread per HVC-I neuron."""
    from unsupervised_growth_amd.engine import Engine
    from unsupervised_growth_amd.network import random_network
    net = random_network(40, 37, n_train=8, p_ra2i=0.5, p_i2ra=0.3, gei_max=2.0, seed=3)
    i = 10241
    padded = dataclasses.replace(net, n_i=i, i2ra_ptr=np.concatenate(
        [net.i2ra_ptr, np.full(i - net.n_i, net.i2ra_ptr[-1], np.int32)]))
    runs = []
    for x in (net, padded):
        with Engine(seed=(5, 0), precision=1, trial_ms=100.0, ra_model=model) as eng:
            eng.upload(x)
            eng.set_tuning(i_lanes=0, ra_lanes=ra_lanes)
            runs.append([eng.run_trial(mode=0, trial_index=k, first_trial=k == 0, mean_injection_time=10.0,
                                       want_state=True) for k in range(2)])
    for a, b in zip(*runs):
        assert sum(map(len, a.interneuron)) > 0
        np.testing.assert_array_equal(a.i_state, b.i_state[:net.n_i])
        np.testing.assert_array_equal(a.ra_state, b.ra_state)
