"""The resident step loop (option 12) at the sizes where it can go wrong, and the
per-step forms it replaces on small networks: bit for bit against the oracle, and
against each other when a network changes between them mid-run."""
import numpy as np
import pytest

from brian2cuda_amd import networks as nw
from brian2cuda_amd import runtime as rt
from test_gpu_networks import ENGINES, _compare

pytestmark = pytest.mark.gpu


def _cuba(n, p, delays, seed=3, we=0.3e-3, wi=-1e-3):
    """n CUBA neurons, random pairs, one weight per pathway, delays drawn from `delays`."""
    rng = np.random.default_rng(seed)
    spec = nw.cuba(N=n, seed=seed, monitors=False)
    ne, paths = max(1, int(0.8 * n)), []
    for var, w, (lo, hi) in ((1, we, (0, ne)), (2, wi, (ne, n))):
        pre, post = np.nonzero(rng.random((hi - lo, n)) < p)
        paths.append(nw.PathSpec(0, 0, var, (pre + lo).astype(np.int32), post.astype(np.int32),
                                 delay_steps=rng.choice(delays, pre.size).astype(np.int32), wmode=0, wscalar=w))
    spec.paths = paths
    spec.spike_monitors = [0]
    spec.state_monitors = [(0, 0, 0, min(n, 5))]
    return spec


def _was_resident(net):
    return net.get_option(rt.OPT_WAS_RESIDENT) == 1


@pytest.mark.parametrize("engine,sem", ENGINES)
@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("n,p,delays", [(1, 1.0, [1]), (2, 1.0, [0]), (63, 0.5, [1]), (64, 0.5, [0, 3]), (65, 0.3, [2]),
                                        (513, 0.1, [1, 2, 3, 40]), (1000, 0.05, [7]), (4097, 0.01, [1]),
                                        (5000, 0.02, [9, 60])])
def test_sizes_and_delays(hs, oracle_lib, n, p, delays, prec, engine, sem):
    """One block and many, ragged last blocks and waves; windows of 1 to 8 steps and
    runs that end inside one; delays shorter and longer than a run."""
    net, _ = _compare(_cuba(n, p, delays), prec, engine, sem, None, oracle_lib, chunks=[20, 1, 11, 3, 300])
    assert _was_resident(net)


@pytest.mark.parametrize("engine,sem", ENGINES)
@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("n,delays", [(1000, [1]), (1000, [3]), (700, [0, 1, 2, 30])])
def test_everyone_fires(hs, oracle_lib, n, delays, prec, engine, sem):
    """All neurons fire in one step: lines of more spikes than a header or a polling
    thread takes, buckets of the plain form that overflow and are delivered from the
    spikes of this launch or of the one before."""
    spec = _cuba(n, 0.5, delays, we=1e-6, wi=-1e-6)
    spec.groups[0].init[0] = np.full(n, -49.5e-3)
    for chunks in ([60, 60], [12, 2, 1, 1, 50]):
        net, ref = _compare(spec, prec, engine, sem, None, oracle_lib, chunks=chunks)
        assert _was_resident(net) and ref.events > 0.4 * n * n


def _weighted(n, degree, by, seed=7):
    """n CUBA neurons, each target with `degree` sources per pathway, a weight of its own per synapse or per source."""
    rng = np.random.default_rng(seed)
    spec, paths = nw.cuba(N=n, seed=seed, monitors=False), []
    for var, scale in ((1, 1.5e-3), (2, -3e-3)):
        pre = np.concatenate([rng.choice(n, degree, replace=False) for _ in range(n)]).astype(np.int32)
        post = np.repeat(np.arange(n, dtype=np.int32), degree)
        w = scale * rng.uniform(0.2, 1.0, pre.size if by == rt.HS_W_SYNAPSE else n)
        o = rng.permutation(pre.size)
        paths.append(nw.PathSpec(0, 0, var, pre[o], post[o], delay_steps=rng.choice([1, 2, 30], pre.size).astype(np.int32),
                                 wmode=by, weights=w))
    spec.paths, spec.spike_monitors, spec.state_monitors = paths, [0], [(0, 0, 0, n)]
    return spec


@pytest.mark.parametrize("by", [rt.HS_W_SYNAPSE, rt.HS_W_PRE])
@pytest.mark.parametrize("engine,sem", ENGINES)
@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("n", [65, 1500, 7001])
def test_weights_of_one_source_each(hs, oracle_lib, n, prec, engine, sem, by):
    """Every synapse's own weight reaches its own target: one source per target and variable, so no two additions meet
    and the bits are the oracle's."""
    net, ref = _compare(_weighted(n, 1, by), prec, engine, sem, None, oracle_lib, chunks=[50, 301, 150])
    assert _was_resident(net) and ref.events > n


@pytest.mark.parametrize("by", [rt.HS_W_SYNAPSE, rt.HS_W_PRE])
@pytest.mark.parametrize("engine,sem", ENGINES)
def test_weights_of_many_sources(hs, oracle_lib, engine, sem, by):
    """The effects of a step on one target are added in any order: at most `degree` additions of a step differ by
    degree eps times their sum of degree times the largest weight; over the steps the synaptic currents only decay, and a
    step adds less than them to v."""
    n, degree, steps = 2000, 40, 400
    spec = _weighted(n, degree, by)
    net, smon, st = nw.build_hs(spec, 64, engine)
    ref, rsmon, rst = oracle_lib.build_ref(spec, 64, sem)
    net.run(steps)
    ref.run(steps)
    assert _was_resident(net) and ref.events > 1000 and net.stats()["events"] == ref.events
    for x, y in zip(net.spikes(smon[0]), ref.spikes(rsmon[0])):
        np.testing.assert_array_equal(x, y)
    atol = steps * degree * np.finfo(np.float64).eps * degree * 3e-3
    for var in (1, 2):
        np.testing.assert_allclose(net.get_state(0, var), ref.get_state(0, var), rtol=0, atol=atol)
    np.testing.assert_allclose(net.state_monitor(st[0], n), ref.state_monitor(rst[0], n), rtol=0, atol=steps * atol)
    net.close()


@pytest.mark.parametrize("opts", [{}, {9: 1}, {9: 1, 4: 2}])
@pytest.mark.parametrize("engine,sem", ENGINES)
@pytest.mark.parametrize("spec", ["brunel", "cuba", "cobahh"])
def test_changes_between_the_forms(hs, oracle_lib, spec, engine, sem, opts):
    """A network that leaves the resident loop and comes back gives the oracle's bits
    throughout, events in flight included."""
    spec = {"brunel": lambda: nw.brunel(N=2000, K=200, seed=4, monitors=True), "cuba": lambda: nw.cuba(N=1500, seed=5),
            "cobahh": lambda: nw.cobahh(N=600, seed=6)}[spec]()
    for prec in (64, 32):
        net, smon, _ = nw.build_hs(spec, prec, engine, options=opts)
        ref, rsmon, _ = oracle_lib.build_ref(spec, prec, sem)
        for k, on in ((40, 0), (300, 1), (33, 0), (1, 1), (2, 0), (250, 1), (200, 0)):
            net.set_option(rt.OPT_RESIDENT, on)
            net.run(k)
            ref.run(k)
            assert _was_resident(net) == bool(on)
            assert net.stats()["events"] == ref.events
            assert np.array_equal(net.get_state(0, 0), ref.get_state(0, 0), equal_nan=True)
        gi, gt = net.spikes(smon[0])
        ri, rtt = ref.spikes(rsmon[0])
        assert len(gi) > 100 and np.array_equal(gi, ri) and np.array_equal(gt, rtt)
        net.close()


def test_layout_waits_for_enough_steps(hs):
    """Many synapses and few steps: the per-step form runs until the steps asked for pay for the layout."""
    spec = nw.brunel(N=4000, K=1000, seed=2, device_connect=True)  # 4e6 synapses: 90 steps
    net, _, _ = nw.build_hs(spec, 32, "fused")
    seen = []
    for _ in range(4):
        net.run(40)
        seen.append(_was_resident(net))
    assert seen == [False, False, True, True]
    net.close()


@pytest.mark.parametrize("n,steps,resident", [(2000, 1534, False), (2000, 1535, True), (1800, 26, False), (1800, 28, True)])
def test_first_run_over_many_synapses(hs, n, steps, resident):
    """Beyond 1e6 synapses the first run has to ask for 1500 steps more than the 10 and one per 50,000 synapses that
    it takes below."""
    net = rt.Net(32, "fused", 1e-4, 1)
    spec = nw.brunel(N=n, K=100, seed=2)
    net.add_group(spec.groups[0].model, n, spec.groups[0].params)
    pid = net.connect_fixed(0, 0, 0, 625 if n == 2000 else 500, delay=(5e-4, 5e-3), w=(-1e-4, -1e-4))
    assert net.pathway_info(pid)["nsyn"] == (1250000 if n == 2000 else 900000)
    net.run(steps)
    assert _was_resident(net) == resident
    net.close()


def test_refuses_nothing_and_leaves_the_rest_alone(hs, oracle_lib):
    """Networks outside the loop's geometry keep running in the per-step forms: more
    neurons than the chip's blocks own, sums that do not fit LDS, several groups."""
    big = nw.brunel(N=140_000, K=10, seed=1, device_connect=True)
    wide = nw.brunel(N=100_000, K=20, seed=1, device_connect=True)
    for spec, prec, engine in ((big, 32, "fused"), (wide, 64, "fused"), (nw.code_mix(N=400, monitors=False), 64, "plain")):
        net, _, _ = nw.build_hs(spec, prec, engine)
        net.run(100)
        assert not _was_resident(net)
        net.close()


@pytest.mark.parametrize("opts", [{}, {9: 1}, {4: 3}, {9: 1, 4: 2, 0: 64, 1: 768, 8: 768}, {0: 128, 1: 512, 10: 256},
                                  {2: 0}])
@pytest.mark.parametrize("engine,sem", ENGINES)
@pytest.mark.parametrize("prec", [64, 32])
def test_per_step_forms_on_small_networks(hs, oracle_lib, prec, engine, sem, opts):
    """The update, delivery, fused and window kernels, which larger networks run."""
    opts = {**opts, rt.OPT_RESIDENT: 0}
    for spec in (nw.brunel(N=2500, K=250, seed=6, monitors=True), nw.cuba(N=1500, seed=5), nw.cobahh(N=600, seed=6)):
        net, _ = _compare(spec, prec, engine, sem, None, oracle_lib, options=opts, chunks=[7, 300, 93])
        assert not _was_resident(net)


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("engine,sem,delay", [("plain", 0, 1), ("plain", 0, 0), ("fused", 1, 0)])
def test_synapse_monitor_between_runs(hs, oracle_lib, engine, sem, delay, prec):
    """A synapse StateMonitor added after a resident run records every step that
    follows: the network goes on in the per-step form, with the oracle's bits."""
    spec = _cuba(300, 0.1, [delay])
    P = spec.paths[0]
    P.wmode, P.weights = rt.HS_W_SYNAPSE, np.full(P.nsyn, P.wscalar)
    net, smon, _ = nw.build_hs(spec, prec, engine)
    ref, rsmon, _ = oracle_lib.build_ref(spec, prec, sem)
    net.run(60)
    assert _was_resident(net)
    which = np.array([5, 0, P.nsyn - 1, 7], np.int32)
    mid = net.add_synapse_monitor(0, rt.HS_SYN_W, which)
    net.run(30)
    net.run(31)
    assert not _was_resident(net)
    w = net.synapse_var(0, rt.HS_SYN_W)[which]
    assert w.min() > 0
    np.testing.assert_array_equal(net.state_monitor(mid, which.size), np.tile(w, (61, 1)))
    ref.run(121)
    assert net.stats()["events"] == ref.events
    for a, b in zip(net.spikes(smon[0]), ref.spikes(rsmon[0])):
        np.testing.assert_array_equal(a, b)
    net.close()


def test_run_time_counts_the_layout(hs):
    """A run that lays the synapses out takes that long: its time is not that of a run after prepare."""
    spec, wall = nw.cuba(N=16000, p=0.003, monitors=False), {}  # 7.7e5 synapses
    for prepared in (False, True):
        for _ in range(6):
            net, _, _ = nw.build_hs(spec, 32, "fused")
            if prepared:
                net.prepare(40)
            net.run(40)
            s = net.stats()
            assert _was_resident(net) and s["last_run_steps"] == 40
            wall[prepared] = min(wall.get(prepared, 1.0), s["last_run_wall_s"])
            net.close()
    assert wall[False] > 1.5 * wall[True]


def _driven(n, degree, mu, delays, seed=5):
    """n noise-driven neurons that fire as mu says, whatever reaches them: `degree` synapses each; mu None: CUBA neurons
    well above their threshold."""
    if mu is None:
        spec = _cuba(n, degree / n, [int(round(d * 1e4)) for d in delays], we=1e-9, wi=-1e-9)
        spec.groups[0].params = [-20e-3, *spec.groups[0].params[1:]]
        spec.state_monitors, spec.rate_monitors = [(0, 0, 0, 7)], [(0, 0, n)]
        return spec
    spec = nw.brunel(N=n, K=degree, seed=seed, J=-1e-9, dlo=delays[0], dhi=delays[1], mu=mu, monitors=True)
    spec.state_monitors, spec.rate_monitors = [(0, 0, 0, 7)], [(0, 0, n)]
    return spec


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("n,degree,mu,delays,engine,sem", [
    (1500, 200, 0.2, (1e-3, 2e-2), "plain", 0), (1500, 200, 0.2, (1e-4, 5e-3), "plain", 0), (700, 100, 0.2, (0.0, 2e-2), "plain", 0),
    (4000, 80, None, (7e-4, 3e-3), "plain", 0), (4000, 80, None, (7e-4, 3e-3), "fused", 1),
    (3000, 100, 0.2, (5e-4, 5e-3), "fused", 1), (3000, 100, 0.2, (2e-4, 3e-4), "fused", 1)])
def test_busy_networks_leave_the_loop(hs, oracle_lib, n, degree, mu, delays, engine, sem, prec):
    """A network that turns out too busy ends its launch early, at the same step in all blocks, and goes on in the per-step
    form with the oracle's bits: spikes, events, monitors, effects in flight."""
    spec = _driven(n, degree, mu, delays)
    for opts in ({}, {9: 1}) if engine == "fused" else ({},):
        net, smon, st = nw.build_hs(spec, prec, engine, options=opts)
        ref, rsmon, rst = oracle_lib.build_ref(spec, prec, sem)
        seen = []
        for k in (20, 1400, 1, 300):
            net.run(k)
            ref.run(k)
            seen.append(_was_resident(net))
            assert net.stats()["events"] == ref.events and net.stats()["steps"] == sum((20, 1400, 1, 300)[:len(seen)])
            assert np.array_equal(net.get_state(0, 0), ref.get_state(0, 0))
        assert seen == [True, False, False, False], seen
        for a, b in zip(net.spikes(smon[0]), ref.spikes(rsmon[0])):
            np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(net.state_monitor(st[0], 7), ref.state_monitor(rst[0], 7))
        np.testing.assert_allclose(net.rate_monitor(net.rate_mids[0]),
                                   np.bincount(ref.spikes(rsmon[0])[1], minlength=1721) / (n * spec.dt), rtol=1e-12)
        net.close()


def test_busy_networks_do_not_enter(hs):
    """The rates of the per-step form keep a network out whose windows hold more than the loop's lists."""
    for mu, resident in ((0.0215, True), (0.2, False)):
        net, _, _ = nw.build_hs(_driven(3000, 100, mu, (5e-4, 5e-3)), 32, "fused", options={rt.OPT_RESIDENT: 0})
        net.run(600)
        net.set_option(rt.OPT_RESIDENT, 1)
        net.run(100)
        assert _was_resident(net) == resident
        net.close()


@pytest.mark.parametrize("engine,sem", ENGINES)
def test_short_runs_with_many_spikes_in_flight(hs, oracle_lib, engine, sem):
    """Single steps of a network whose delays hold 1700 spikes, which the loop's start would deliver again, take the
    per-step form; longer runs the loop; the bits are the oracle's throughout."""
    spec = _driven(8000, 50, 0.025, (5e-4, 5e-3))
    net, smon, _ = nw.build_hs(spec, 64, engine)
    ref, rsmon, _ = oracle_lib.build_ref(spec, 64, sem)
    seen = []
    for k in (300, 1, 1, 50, 1, 120):
        net.run(k)
        ref.run(k)
        seen.append(_was_resident(net))
        assert net.stats()["events"] == ref.events and np.array_equal(net.get_state(0, 0), ref.get_state(0, 0))
    assert seen == [True, False, False, True, False, True], seen
    for a, b in zip(net.spikes(smon[0]), ref.spikes(rsmon[0])):
        np.testing.assert_array_equal(a, b)
    net.close()


def test_busy_for_a_while(hs):
    """A network that left the loop comes back once it is quiet, after 1000 steps at the earliest."""
    net, _, _ = nw.build_hs(_driven(1500, 300, 0.015, (1e-3, 2e-2)), 64, "plain")
    ref, _, _ = nw.build_hs(_driven(1500, 300, 0.015, (1e-3, 2e-2)), 64, "plain", options={rt.OPT_RESIDENT: 0})
    seen = []
    for x in (net, ref):
        x.set_state(0, 0, np.full(1500, 25e-3))  # everyone fires at once, and rarely after that
    for k in (20, 500, 400, 400, 300, 50):
        for x in (net, ref):
            x.run(k)
        seen.append(_was_resident(net))
        assert net.stats()["events"] == ref.stats()["events"] and net.stats()["spikes"] == ref.stats()["spikes"]
        np.testing.assert_array_equal(net.get_state(0, 0), ref.get_state(0, 0))
    assert seen == [True, False, False, False, True, True], seen
    net.close()
    ref.close()
