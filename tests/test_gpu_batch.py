"""Batched form: several networks of different sizes in one context.

Each network's noise streams are keyed by its own seed and its own neuron ids,
and every ordered sum runs over its own neurons only, so network b of a batch
must produce exactly what a context holding network b alone produces -- spike
trains, neuron states, weights, active / super lists -- in both precision
forms.  The FP64 single-network form is itself bit-exact with the oracle
(test_gpu_parity.py), so this pins the batch to the oracle as well.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _nets():
    from unsupervised_growth_amd.network import random_network
    sizes = [(40, 10, "dense"), (25, 7, 8), (60, 16, 12), (33, 9, "dense")]
    return [random_network(nra, ni, n_train=6, p_ra2i=0.3, p_i2ra=0.3, gie_max=1.0, gei_max=0.5,
                           spread_max=20.0, seed=11 + k, rr=rr) for k, (nra, ni, rr) in enumerate(sizes)]


def _trial(b, tr, mode=0):
    return dict(mode=mode, training=True, trial_index=tr + 3 * b, first_trial=(tr == 0),
                mean_injection_time=100.0 + 7 * b + 3 * tr)


def _same(a, b, what):
    assert len(a) == len(b), what
    for x, y in zip(a, b):
        np.testing.assert_array_equal(np.asarray(x), np.asarray(y), err_msg=what)


@pytest.mark.parametrize("precision", [0, 1])
def test_batch_equals_each_network_alone(precision):
    from unsupervised_growth_amd.engine import Engine
    nets = _nets()
    keys = [(100 + b, 7) for b in range(len(nets))]
    trial_ms = 250.0
    print("batch precision=%d sizes=%s" % (precision, [(n.n_ra, n.n_i) for n in nets]), flush=True)
    alone = []
    for b, net in enumerate(nets):
        with Engine(precision=precision, trial_ms=trial_ms, seed=keys[b]) as e:
            e.upload(net)
            res = [e.run_trial(**_trial(b, tr)) for tr in range(3)]
            syn = e.download_synapses()
            res.append(e.run_trial(**_trial(b, 3, mode=1)))
            alone.append((res, syn))
    with Engine(precision=precision, trial_ms=trial_ms) as e:
        e.upload_batch(nets, keys)
        batch = [e.run_batch([_trial(b, tr) for b in range(len(nets))]) for tr in range(3)]
        syns = [e.download_synapses(b) for b in range(len(nets))]
        batch.append(e.run_batch([_trial(b, 3, mode=1) for b in range(len(nets))]))
    spikes = 0
    for b in range(len(nets)):
        res, syn = alone[b]
        for tr in range(4):
            for kind in ("soma", "dend", "interneuron"):
                _same(getattr(batch[tr][b], kind), getattr(res[tr], kind), "net %d trial %d %s" % (b, tr, kind))
            spikes += sum(map(len, res[tr].soma))
        for k in ("w", "act_cnt", "act_ids", "sup_cnt", "sup_ids", "remodeled"):
            np.testing.assert_array_equal(getattr(syns[b], k), getattr(syn, k), err_msg="net %d %s" % (b, k))
    assert spikes > 0


@pytest.mark.parametrize("precision", [0, 1])
def test_launch_shapes_do_not_change_results(precision):
    """Every launch shape the autotuner may pick gives the same bits (RK4 form),
    the delivery on its lists or sweeping every neuron.  (In FP64 the shapes'
    HVC-RA layouts are one at this size, and i_lanes 1 to 3 are at any;
    test_gpu_octet.py runs the layouts of large networks.)"""
    from unsupervised_growth_amd.engine import Engine
    nets = _nets()
    keys = [(100 + b, 7) for b in range(len(nets))]
    shapes = [dict(integrate_block=64, i_lanes=1, deliver_block=64, sync_block=256, ra_lanes=1, deliver_lists=1),
              dict(integrate_block=256, i_lanes=0, deliver_block=128, sync_block=512, ra_lanes=0, deliver_lists=0),
              dict(integrate_block=128, i_lanes=2, deliver_block=256, sync_block=128, ra_lanes=0, deliver_lists=1),
              dict(integrate_block=256, i_lanes=1, deliver_block=64, sync_block=256, ra_lanes=1, deliver_lists=0),
              dict(integrate_block=64, i_lanes=2, deliver_block=128, sync_block=512, ra_lanes=1, deliver_lists=0),
              dict(integrate_block=128, i_lanes=3, deliver_block=64, sync_block=256, ra_lanes=1, deliver_lists=1),
              dict(integrate_block=256, i_lanes=3, deliver_block=128, sync_block=256, ra_lanes=0, deliver_lists=0),
              dict(integrate_block=256, i_lanes=3, deliver_block=256, sync_block=256, ra_lanes=0, deliver_lists=1)]
    runs = []
    for shape in shapes:
        # the RK4 form for HVC-RA, where FP32 has four lanes per neuron
        with Engine(precision=precision, trial_ms=200.0, ra_model=1) as e:
            e.upload_batch(nets, keys)
            e.set_tuning(**shape)
            assert e.tuning() == shape
            res = [e.run_batch([_trial(b, tr) for b in range(len(nets))]) for tr in range(2)]
            res.append(e.run_batch([_trial(b, 2, mode=1) for b in range(len(nets))]))
            runs.append((res, [e.download_synapses(b) for b in range(len(nets))]))
    for res, syns in runs[1:]:
        for tr in range(3):
            for b in range(len(nets)):
                for kind in ("soma", "dend", "interneuron"):
                    _same(getattr(res[tr][b], kind), getattr(runs[0][0][tr][b], kind), "trial %d net %d" % (tr, b))
        for b in range(len(nets)):
            np.testing.assert_array_equal(syns[b].w, runs[0][1][b].w)


def test_autotune_keeps_a_valid_shape_and_results():
    from unsupervised_growth_amd.engine import Engine
    nets = _nets()
    keys = [(100 + b, 7) for b in range(len(nets))]
    with Engine(precision=1, trial_ms=200.0) as e:
        e.upload_batch(nets, keys)
        ref = e.run_batch([_trial(b, 0, mode=1) for b in range(len(nets))])
        shape, ms = e.autotune(windows=60)
        print("autotune:", shape, ms, flush=True)
        assert shape["integrate_block"] in (64, 128, 256) and shape["deliver_block"] in (64, 128, 256)
        assert shape["sync_block"] in (128, 256, 512) and np.all(ms > 0)
        assert shape["i_lanes"] in (0, 1, 2, 3) and shape["ra_lanes"] in (0, 1)
        again = e.run_batch([_trial(b, 0, mode=1) for b in range(len(nets))])
    for b in range(len(nets)):
        for kind in ("soma", "dend", "interneuron"):
            _same(getattr(again[b], kind), getattr(ref[b], kind), "net %d %s" % (b, kind))


def test_large_batch_pushes_equal_each_network_alone():
    """A batch above 65 536 neurons delivers its fixed-weight edges with one lane
    per presynaptic neuron, a network alone with a quad per neuron: same bits."""
    from unsupervised_growth_amd import configs
    from unsupervised_growth_amd.engine import Engine
    nets = [configs.sphere_network(np.random.default_rng(41 + b), 18000, 5000, 10.0, k_rr=16, n_train=60,
                                   spread_max=20.0) for b in range(3)]
    assert sum(n.n_ra + n.n_i for n in nets) > 65536 and all(n.n_ra + n.n_i <= 65536 for n in nets)
    keys = [(300 + b, 5) for b in range(len(nets))]
    trial_ms = 150.0
    trials = [dict(mode=0, training=True, trial_index=b, first_trial=True, mean_injection_time=40.0 + 5 * b)
              for b in range(len(nets))]
    print("large batch sizes=%s" % [(n.n_ra, n.n_i) for n in nets], flush=True)
    alone = []
    for b, net in enumerate(nets):
        with Engine(precision=1, trial_ms=trial_ms, seed=keys[b]) as e:
            e.upload(net)
            alone.append((e.run_trial(**trials[b]), e.download_synapses()))
    with Engine(precision=1, trial_ms=trial_ms) as e:
        e.upload_batch(nets, keys)
        batch = e.run_batch(trials)
        syns = [e.download_synapses(b) for b in range(len(nets))]
    spikes = 0
    for b in range(len(nets)):
        res, syn = alone[b]
        for kind in ("soma", "dend", "interneuron"):
            _same(getattr(batch[b], kind), getattr(res, kind), "net %d %s" % (b, kind))
        spikes += sum(map(len, res.interneuron))
        np.testing.assert_array_equal(syns[b].w, syn.w, err_msg="net %d w" % b)
    assert spikes > 0
