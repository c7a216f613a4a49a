"""GPU: the spring chains' group kernels at the sizes where a size class or a
lane's masses end.  The methods beside DOPRI5 give the CPU restatement's values
(as the one-lane mapping does); DOPRI5's shapes agree with one another."""
import numpy as np
import pytest

import deamd
from deamd import DE_MAP_AUTO, DE_MAP_GROUP, DE_MAP_LANE, IVP, ExplicitRungeKutta, SpringChain
from test_spring_classes import classes_of

pytestmark = pytest.mark.gpu

THREADS = 8
ADAPTIVE = ["dop853", "rkf45", "cash_karp", "rkv655e", "rkv656e", "rkv766e", "rkv767e", "rkv877e",
            "rkv878e", "rkv988e", "rkv989e"]
FIXED = ["rk4", "euler"]
# One below, at and above every class bound, odd remainders inside the classes
# of two and four masses per lane, and a lone mass.
EDGES = [1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 66, 95, 96, 97, 127, 128,
         129, 130, 131, 191, 192, 193, 254, 255, 256]


def chains(sizes, seed):
    sizes = np.asarray(sizes, dtype=np.int32)
    rng = np.random.default_rng(seed)
    params, y0 = [], []
    for n in sizes:
        params += [rng.uniform(0.0, 0.1, 1), np.exp(0.5 * rng.standard_normal(n + 1))]
        y0 += [rng.standard_normal(n), 0.1 * rng.standard_normal(n)]
    return SpringChain(sizes, np.concatenate(params)), np.concatenate(y0)


def make(method, rtol=1e-7, h=0.01):
    M = ExplicitRungeKutta
    if method in FIXED:
        return getattr(M, method)(h).max_steps(200000)
    return getattr(M, method)().rtol(rtol).atol(rtol * 1e-2).max_steps(200000)


# AUTO solves these small ensembles of many sizes with 64 lanes per system; GROUP with a
# group_size solves each class in its own shape, several systems per wavefront.
BOTH = (DE_MAP_AUTO, DE_MAP_GROUP)


def check(orc, ens, mappings=(DE_MAP_AUTO,)):
    # Equal values, NaN where the oracle has NaN; a zero's sign may differ in
    # the embedded family, whose kernels skip zero coefficients.
    want = orc.solve_ode(ens, threads=THREADS)
    for mapping in mappings:
        got = ens.options(mapping=mapping, group_size=8 if mapping == DE_MAP_GROUP else 0).solve()
        for f in ("status", "accepted", "rejected", "evals"):
            assert np.array_equal(getattr(got, f), getattr(want, f)), (f, mapping)
        for f in ("t", "y", "dense", "n_dense"):
            g, w = getattr(got, f), getattr(want, f)
            assert (g is None) == (w is None)
            if g is not None:
                assert np.array_equal(g, w, equal_nan=g.dtype.kind == "f"), (f, mapping)
    return want


@pytest.mark.parametrize("method", ADAPTIVE + FIXED)
def test_class_edges(orc, method):
    sysm, y0 = chains(EDGES, 71)
    base = lambda: IVP.ode(sysm, 0.0, 1.5, y0).method(make(method))  # noqa: E731
    check(orc, base(), (DE_MAP_AUTO, DE_MAP_GROUP, DE_MAP_LANE))
    # t0, the end and points off both ends among the output times.
    check(orc, base().t_eval(np.concatenate([np.linspace(-0.2, 1.7, 17), [0.0, 1.5]])), BOTH)


@pytest.mark.parametrize("method", ["rk4", "dop853", "rkf45", "rkv767e"])
def test_spans_tolerances_and_statuses(orc, method):
    # Per-system spans (forward, backward, empty: BadInput), per-component and
    # per-system tolerances, and a step limit that some systems reach.
    rng = np.random.default_rng(72)
    sizes = rng.integers(1, 257, 90)
    sysm, y0 = chains(sizes, 73)
    n, state = len(sizes), int(2 * sizes.sum())
    t0 = rng.uniform(-1.0, 1.0, n)
    tf = t0 + rng.uniform(0.2, 2.0, n)
    tf[::9] = t0[::9]
    if method not in FIXED:
        tf[1::3] = t0[1::3] - 0.7
    ens = IVP.ode(sysm, t0, tf, y0).method(make(method).max_steps(60))
    ens.rtol_traj = np.where(np.arange(n) % 2 == 0, 1e-5, 1e-8)
    ens.atol_traj = ens.rtol_traj * 1e-2
    want = check(orc, ens, BOTH + (DE_MAP_LANE,))
    assert set(want.status) >= {deamd.DE_STATUS_COMPLETE, deamd.DE_STATUS_BAD_INPUT}
    ens.rtol_comp = 10.0 ** rng.uniform(-8, -5, state)
    ens.atol_comp = ens.rtol_comp * 1e-2
    check(orc, ens, BOTH)
    # Backward with output: the solve ends at its first interior point.
    back = IVP.ode(sysm, 0.0, -1.0 if method not in FIXED else 1.0, y0).method(
        make(method)).t_eval(np.linspace(0.0, -1.0, 5) if method not in FIXED else [0.5])
    check(orc, back, BOTH)


@pytest.mark.parametrize("method", ["dop853", "rkf45", "rkv877e"])
def test_values_that_overflow(orc, method):
    # Springs stiff enough that stages overflow: rejections, NaN where the
    # reference's combinations give NaN, and the stiffness and step-size ends.
    sysm, y0 = chains([1, 4, 3, 4, 5, 7, 12, 16, 33, 64, 65, 129, 200, 2], 74)
    p = sysm.params_packed.copy()
    for i in range(0, len(sysm.sizes), 2):
        lo = int(sysm.param_offset[i])
        p[lo + 1:lo + 2 + int(sysm.sizes[i])] = 1e200
    y0 = y0.copy()
    y0[-3] = np.inf
    ens = IVP.ode(SpringChain(sysm.sizes, p), 0.0, 1.0, y0).method(
        make(method).h0(0.1).max_steps(500).max_rejects(7))
    check(orc, ens, BOTH + (DE_MAP_LANE,))


@pytest.mark.parametrize("method,sizes", [("dopri5", (300, 6144, 6145, 16384)),
                                          ("dop853", (300, 12289)), ("rk4", (300, 12289))])
def test_results_do_not_depend_on_the_batch(orc, method, sizes):
    # The classes that a launch uses follow its systems; a system has the same bits
    # alone and in an ensemble of every set of classes.
    edges = [6, 23, 40, 100, 160, 200, 3, 64]
    rng = np.random.default_rng(75)
    pool = np.concatenate([edges, rng.integers(1, 33, 92)])
    sysm, y0 = chains(pool, 75)

    def part(idx):
        so, po = sysm.state_offset, sysm.param_offset
        p = np.concatenate([sysm.params_packed[po[i]:po[i + 1]] for i in idx])
        y = np.concatenate([y0[so[i]:so[i + 1]] for i in idx])
        return IVP.ode(SpringChain(pool[idx], p), 0.0, 0.6, y).method(make(method, h=0.02))

    alone = [part([i]).solve() for i in range(len(edges))]
    if method != "dopri5":
        assert all(np.array_equal(a.y, orc.solve_ode(part([i])).y) for i, a in enumerate(alone))
    sets = set()
    for n in sizes:
        idx = np.concatenate([np.arange(len(edges)), rng.integers(0, len(pool), n - len(edges))])
        sets.add(classes_of(method == "dopri5", pool[idx]))
        whole = part(idx).solve()
        for i, one in enumerate(alone):
            assert np.array_equal(one.y, whole.final_state(i)), (n, i)
            assert one.accepted[0] == whole.accepted[i] and one.evals[0] == whole.evals[i]
    assert sets == ({"few", "mid", "all"} if method == "dopri5" else {"few", "all"})


@pytest.mark.parametrize("out", ["final", "t_eval", "points", "event"])
def test_dopri5_shapes_agree(orc, out):
    # Every shape (lanes per system, masses per lane) of a size class adds the
    # norm in one order, so the shape does not change a bit; against the oracle
    # the sums' order and the fused interpolant leave roundings (the group
    # mappings' bound: final state within 1e-10 of the state's largest value).
    sysm, y0 = chains(EDGES, 76)
    ens = IVP.ode(sysm, 0.0, 3.0, y0).method(make("dopri5"))
    if out == "t_eval":
        ens = ens.t_eval(np.linspace(-0.1, 3.0, 14))
    elif out == "points":
        ens = ens.even(0.21)
    elif out == "event":
        ens = ens.event(deamd.Event.component(0, 0.05))
    want = orc.solve_ode(ens, threads=THREADS)
    first = ens.options(mapping=DE_MAP_AUTO, group_size=0).solve()
    for f in ("status", "accepted", "rejected", "evals"):
        assert np.array_equal(getattr(first, f), getattr(want, f)), f
    for i in range(len(EDGES)):
        w = want.final_state(i)
        assert np.abs(first.final_state(i) - w).max() <= 1e-10 * np.abs(w).max()
    for g in (1, 2, 4, 8, 16, 32, 64):
        got = ens.options(mapping=DE_MAP_GROUP, group_size=g).solve()
        for f in ("status", "accepted", "rejected", "evals", "t", "y", "dense", "n_dense",
                  "n_events", "n_points"):
            a, b = getattr(got, f), getattr(first, f)
            assert (a is None) == (b is None)
            if a is not None:
                assert np.array_equal(a, b, equal_nan=a.dtype.kind == "f"), (f, g)
        if out == "points":
            for i in range(len(EDGES)):
                for a, b in zip(got.points(i), first.points(i)):
                    assert np.array_equal(a, b)
        if out == "event":
            assert np.array_equal(got.event_t, first.event_t, equal_nan=True)
            assert np.array_equal(got.event_y, first.event_y, equal_nan=True)


def test_stiffness_end(orc):
    # The reference's stiffness test compares |yseg - k| with |f(y_new) - y_stage|; for
    # f(y) = y (no springs, damping -1, v = x) the second is rounding-level, so that the
    # solves end by it; with damping -0.6 they go on.
    sysm, y0 = chains([1, 2, 3, 4, 4, 3, 6, 8, 13, 30, 60, 120, 250] * 2, 77)
    rng = np.random.default_rng(77)
    p = np.zeros_like(sysm.params_packed)
    n = len(sysm.sizes)
    p[sysm.param_offset[:-1]] = np.where(np.arange(n) < n // 2, -1.0, -0.6)
    for i, m in enumerate(sysm.sizes):
        lo = int(sysm.state_offset[i])
        y0[lo:lo + m] = y0[lo + m:lo + 2 * m] = rng.uniform(0.5, 2.0, m)
    ens = IVP.ode(SpringChain(sysm.sizes, p), 0.0, rng.uniform(22.0, 30.0, n), y0).method(
        make("dop853", rtol=1e-12).h0(0.005).h_max(0.01))
    want = check(orc, ens, BOTH + (DE_MAP_LANE,))
    assert (want.status == deamd.DE_STATUS_STIFFNESS).sum() >= n // 3
    assert (want.status == deamd.DE_STATUS_COMPLETE).sum() >= n // 3
