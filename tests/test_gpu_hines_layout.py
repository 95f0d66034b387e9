"""Multicompartment batches at the edges of the kernel's split: sections around
the 64 lanes of a solver wave, nodes around its registers, sections of unequal
length, trees per compute unit around the rule for waves and LDS, and values that
the short divisions do not cover (potentials, time step, numerators next to zero).
Bit for bit against the oracle."""
import numpy as np
import pytest

import oracle
from brian2cuda_amd import morphology as mo

pytestmark = pytest.mark.gpu


def _combs(sizes, n_trees=1, dt=0.025e-3, d=1e-6, l=30e-6):
    """n_trees trees: a main path of the even sections, a side branch (odd) from each; section s has sizes[s]."""
    ns, nc = len(sizes), int(np.sum(sizes))
    parent = [-1] + [s - 1 if s % 2 else s - 2 for s in range(1, ns)]
    rng = np.random.default_rng([ns, nc, n_trees])
    cur = np.zeros(nc * n_trees)
    cur[::nc] = rng.uniform(0.1e-9, 1e-9, n_trees)
    n = nc * n_trees
    rl = np.full(n, np.pi * d * d / (2 * l))
    return mo.TreeBatch(
        dt, np.arange(n_trees + 1, dtype=np.int32) * nc, np.arange(n_trees + 1, dtype=np.int32) * ns,
        np.tile(np.cumsum([0] + list(sizes[:-1])).astype(np.int32), n_trees), np.tile(np.array(sizes, np.int32), n_trees),
        np.tile(np.array(parent, np.int32), n_trees), np.full(n, np.pi * d * l), rl, rl.copy(), np.full(n, 1e-2),
        init={0: rng.uniform(-0.02, 0.02, n), 1: np.full(n, 0.05), 2: np.full(n, 0.32), 3: np.full(n, 0.6), 4: cur})


def _check(tb, prec, steps):
    g, r = mo.build_hs(tb, prec), oracle.RefMC(tb, prec)
    g.run(steps)
    r.run(steps)
    for var in range(4):
        np.testing.assert_array_equal(g.get_state(var), r.get_state(var), err_msg=f"var {var}")
    np.testing.assert_array_equal(g.spike_counts(), r.spike_counts())


@pytest.mark.parametrize("ns", [1, 2, 63, 64, 65, 127, 128, 129, 192, 193, 255])
def test_sections_and_nodes(hs, ns):
    _check(_combs([1 + s % 4 for s in range(ns)], n_trees=3), 64, 60)


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("sizes", [[1], [2], [3, 1, 40], [1, 5, 300, 2, 1], [1024], [16] * 64, [4] * 255])
def test_section_lengths(hs, sizes, prec):
    _check(_combs(sizes, n_trees=2), prec, 60)


@pytest.mark.parametrize("n_trees", [255, 257, 513, 1300, 4100])
def test_trees_per_unit(hs, n_trees):
    _check(_combs([3, 2, 9, 4, 1], n_trees), 64, 40)


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("kind", ["potential", "step", "weak", "gates", "negative", "nan"])
def test_outside_the_short_forms(hs, kind, prec):
    tb = _combs([4, 3, 200], n_trees=3, dt=0.1e-3 if kind == "step" else 0.025e-3, l=3e-3 if kind == "weak" else 30e-6)
    if kind == "potential":
        tb.init[0][7] = 0.3
        tb.init[0][tb.n_comp // 2] = -0.2
    if kind == "weak": # each compartment sees about 1e-6 of its neighbour: 200 of them reach below the smallest double
        tb.init[0][:] = 0
    if kind == "gates": # two conductances whose sum leaves the exponent range, their currents do not: a row divides by infinity
        most = 1.6e308 if prec == 64 else 3e38
        for i in (5, tb.n_comp // 2):
            tb.init[1][i], tb.init[2][i] = (most / tb.chan[2]) ** (1 / 3), (0.8 * most / tb.chan[4]) ** 0.25
    if kind == "negative": # a diagonal of either sign
        tb.init[3][9:12] = [-1e3, -0.05, -1e-3]
    if kind == "nan":
        tb.init[1][5] = np.nan
    _check(tb, prec, 40)


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("sizes,n_trees", [([5, 1, 30, 2], 3), ([16] * 40, 520)])
def test_state_between_launches(hs, sizes, n_trees, prec):
    """The caller's order of the compartments between launches of a few steps, with the gates of a launch in LDS (3 trees)
    and in global memory (520 of 640 compartments): states and currents set and read in between."""
    tb = _combs(sizes, n_trees)
    g, r = mo.build_hs(tb, prec), oracle.RefMC(tb, prec)
    g.set_option(0, 3)
    rng = np.random.default_rng(9)
    for k in range(2):
        g.run(7)
        r.run(7)
        for var in range(4):
            np.testing.assert_array_equal(g.get_state(var), r.get_state(var), err_msg=f"var {var}")
        for var, new in ((0, rng.uniform(-0.02, 0.02, tb.n_comp)), (2, rng.uniform(0, 1, tb.n_comp)),
                         (4, rng.uniform(0, 1e-11, tb.n_comp))):
            g.set_state(var, new)
            r.set_state(var, new)
            if var != 2:
                np.testing.assert_array_equal(g.get_state(var), new)
