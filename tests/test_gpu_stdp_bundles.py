"""on_pre of STDP pathways where its rules and its 256-thread rounds turn over: few
spikes, spikes of one step around 256, groups whose spikes go to several lists,
bundles from nothing to more synapses than threads and around the mean size from
which they are taken one after another, many spikes on one target.  Synapse variables bit for
bit against the oracle's sequential loop, the targets' state too where the order of
the spikes is its order, else within the rounding of the sums."""
import numpy as np
import pytest

from brian2cuda_amd import networks as nw
from brian2cuda_amd import runtime as rt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("n_in,n_out,degree", [(1, 1, 1), (255, 3, 1), (256, 1, 1), (257, 2, 2), (700, 3, 1), (5, 257, 257),
                                               (3, 900, 600), (520, 40, 0), (2, 90, 64), (40, 50, 6), (40, 50, 7),
                                               (300, 50, 6), (300, 50, 7), (140000, 2, 1), (132000, 9, 8)])
def test_bursts_vs_oracle(hs, oracle_lib, n_in, n_out, degree, prec):
    rs = np.random.RandomState(n_in + n_out)
    steps = np.array([2, 3, 40, 41, 90])
    src, t = [], []
    for k, s in enumerate(steps): # everyone, then random subsets
        who = np.arange(n_in) if k in (0, 3) else np.flatnonzero(rs.rand(n_in) < 0.6)
        src.append(who)
        t.append(np.full(who.size, s))
    G = nw.GroupSpec(rt.HS_MODEL_SPIKEGEN, n_in, [0.0],
                     spikes=(np.concatenate(src).astype(np.int32), np.concatenate(t).astype(np.int64)))
    P = nw.GroupSpec(rt.HS_MODEL_LIF_CUBA, n_out, [-49e-3, -50e-3, -60e-3, 20e-3, 5e-3, 5e-3, 5e-3, 1.0],
                     {0: -60e-3 + 10e-3 * rs.rand(n_out), 1: 0.0})
    kids = [rs.choice(n_out, degree or rs.randint(0, n_out + 1), replace=False) for _ in range(n_in)]
    ii = np.repeat(np.arange(n_in), [k.size for k in kids]).astype(np.int32)
    S = nw.PathSpec(0, 1, 1, ii, np.concatenate(kids).astype(np.int32), scalar_delay=0, wmode=rt.HS_W_SYNAPSE,
                    weights=1.5 + 2.0 * rs.rand(ii.size), stdp=(20e-3, 20e-3, 0.05, -0.055, 0.0, 4.0, 1e-3))
    spec = nw.NetSpec("stdp_bursts", 0.1e-3, 1, [G, P], [S], spike_monitors=[1], state_monitors=[(1, 0, 0, n_out)])
    net, sm, st = nw.build_hs(spec, prec, "plain")
    ref, rsm, rst = oracle_lib.build_ref(spec, prec, oracle_lib.SEQ)
    net.run(120)
    ref.run(120)
    perm = np.argsort(ii, kind="stable")
    for var in (rt.HS_SYN_W, rt.HS_SYN_APRE, rt.HS_SYN_APOST, rt.HS_SYN_LASTUPDATE):
        a, b = net.synapse_var(0, var), ref.synapse_var(0, var, S.nsyn)
        np.testing.assert_array_equal(np.sort(a), np.sort(b[perm]), err_msg=str(var))
    # a step's spike list is in the order in which waves append to it, and a bundle's synapses are spread over waves, so a
    # target's additions come in another order than the loop's where several waves spike or share a bundle: m additions of
    # at most 4 mV differ by at most m eps times their sum of m 4 mV per burst, and the leak only shrinks it
    m = n_in if n_in > 64 or degree > 64 else 0
    eps = np.finfo(np.float64 if prec == 64 else np.float32).eps
    np.testing.assert_allclose(net.state_monitor(st[0], n_out), ref.state_monitor(rst[0], n_out), rtol=0,
                               atol=steps.size * m * eps * m * 4e-3)
    assert net.stats()["events"] == ref.events
    net.close()
