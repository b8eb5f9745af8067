"""The persistent row kernel (one pulse, whole runs in one cooperative
launch) against the same run with one launch per stage, which sums in the
same order, so the two agree bit for bit; and its way back when a launch
gives up waiting.  The shapes sit at the kernel's edges: single states, row
counts around the quads of 4 and workgroups of 16, neighbour columns around
the 64-column chunks and the 16 chunks held in registers, chunks in LDS and
past it, and more than 16 and 32 rows a workgroup."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [[1, 1], [3, 2, 4], [17, 64, 65, 5], [63, 129, 1, 16],
          [300, 257, 513], [511, 513, 40], [1025, 30, 1100],
          [2300, 9, 2600, 3], [4100, 8, 2100], [9000, 2, 3]]


@pytest.fixture(scope="module")
def mpci():
    import mpci as m
    assert m.device_count() >= 1
    return m


def state(n, seed):
    x = np.random.default_rng(seed).standard_normal(2 * n)
    return x / np.linalg.norm(x)


def make(mpci, g, x0, graph, gauge):
    prop = mpci.Propagator(g)
    assert prop.set_small_path(1)
    prop.set_graph(graph)
    prop.set_state(x0)
    prop.set_pulse(mpci.Pulse.sine(0.04 ** 2, 0.7, 2, gauge))
    return prop


@pytest.mark.parametrize("gauge", ["v", "l"])
@pytest.mark.parametrize("s", SHAPES)
def test_persistent_equals_stage_launches(mpci, s, gauge):
    from mpci import synth
    E, D = synth.system_arrays(s, seed=sum(s))
    g = mpci.System(E, D, gauge=gauge)
    x0 = state(g.N, len(s))
    F = 0.05 * np.sin(np.arange(9.0))[None]
    runs = []
    for graph in (True, False):
        prop = make(mpci, g, x0, graph, gauge)
        # the first trial steps of 2 a.u. are rejected
        st, log = prop.prop_adaptive(3.0, 7.0, 2.0, 1e-9, 1e-9, track=g.N - 1,
                                     log_cap=400)
        xa = prop.get_state()
        pop = prop.prop_fixed(0.0, 0.1, F, track=g.N // 2)
        prop.prop_schedule(1.0, [[0.1, 0.2, 0.05]])
        runs.append((st[0].accepted, st[0].rejected, st[0].t, st[0].h, log,
                     xa, pop, prop.get_state()))
        prop.close()
    assert runs[0][1] >= 1
    for a, b in zip(*runs):
        assert np.array_equal(a, b)


# around the units of 128 x 256, the 16-row groups, one and two segments a
# workgroup, groups in registers, in LDS and streamed, narrow column blocks
TILE_SHAPES = [[1777, 2401], [2049, 2100, 16], [40, 13000, 257],
               [300, 6200, 1100], [2400, 2500, 1300], [1, 4200, 3],
               [9] * 28 + [1300, 2500]]


@pytest.mark.parametrize("gauge", ["v", "l"])
@pytest.mark.parametrize("s", TILE_SHAPES)
def test_persistent_tiles_against_oracle(mpci, oracle, s, gauge):
    """The persistent tile kernel (larger systems): two frozen-field steps
    against the oracle within 1e-12, the run split in two calls bit for bit,
    the adaptive mode's counts against stage launches (another summation
    order: the state within 1e-11), and the way back when a launch gives up."""
    from mpci import synth
    E, D = synth.system_arrays(s, seed=sum(s))
    g, o = mpci.System(E, D, gauge=gauge), oracle.System(E, D, gauge=gauge)
    # past the row form's range
    assert sum(-(-n // 16) for n in s) > 256
    x0 = state(g.N, 7)
    F = np.array([[0.04, -0.03, 0.02]])

    def prop(graph=True):
        p = mpci.Propagator(g)
        p.set_graph(graph)
        p.set_state(x0)
        p.set_pulse(mpci.Pulse.sine(0.04 ** 2, 0.7, 2, gauge))
        return p

    a = prop()
    a.prop_fixed(0.0, 0.1, F)
    xr = x0.copy()
    for k in range(3):
        xr = o.step(F[0, k], xr, 0.1)
        xr /= np.sqrt(xr @ xr)
    assert np.abs(a.get_state() - xr).max() < 1e-12
    b = prop()
    b.prop_fixed(0.0, 0.1, F[:, :1])
    b.prop_fixed(0.1, 0.1, F[:, 1:])
    assert np.array_equal(a.get_state(), b.get_state())
    b.set_state(x0)
    b.set_wait_limit(-1)
    b.prop_fixed(0.0, 0.1, F)
    assert np.abs(a.get_state() - b.get_state()).max() < 1e-14
    c = prop(False)
    a.set_state(x0)
    st = [p.prop_adaptive(3.0, 6.0, 1.5, 1e-9, 1e-9)[0][0] for p in (a, c)]
    assert st[0].accepted == st[1].accepted and st[0].rejected >= 1
    assert st[0].rejected == st[1].rejected
    assert np.abs(a.get_state() - c.get_state()).max() < 1e-11


# one and several pulses a group, groups with a pulse less, a workgroup's
# eight slots used up (nine pulses a group of the blocks 950, 2, 2, ..)
@pytest.mark.parametrize("s,P", [([1, 1], 2), ([17, 64, 65, 5], 3),
                                 ([60, 72, 48], 100), ([300] * 6, 5),
                                 ([250] * 16, 3), ([950] + [2] * 20, 26),
                                 ([2000, 2000], 2)])
def test_batch_equals_single_pulses(mpci, s, P):
    """A batch in the persistent row form: every pulse equals its own run
    alone bit for bit, pulses that end at different times, one of no length
    and one with rejected steps among them; and equals the batched launches
    to rounding (1e-12), also after a launch gave up."""
    from mpci import synth
    E, D = synth.system_arrays(s, seed=sum(s))
    g = mpci.System(E, D)
    xs = [state(g.N, 50 + p) for p in range(P)]
    F = 0.05 * np.sin(np.arange(7.0) + np.arange(P)[:, None])
    t1 = 3.0 + 0.3 * (np.arange(P) % 7)
    t1[P // 2] = 1.0
    h0 = np.where(np.arange(P) == 0, 2.0, 0.1)

    def run(ps, graph=True, ms=0):
        prop = mpci.Propagator(g, P=len(ps))
        prop.set_graph(graph)
        for i, p in enumerate(ps):
            prop.set_state(xs[p], i)
            prop.set_pulse(mpci.Pulse.sine(0.04 ** 2, 0.5 + 0.01 * p, 2), i)
        prop.set_wait_limit(ms)
        pop = prop.prop_fixed(0.0, 0.1, F[ps], track=g.N // 2)
        x1 = [prop.get_state(i) for i in range(len(ps))]
        st, log = prop.prop_adaptive(1.0, t1[ps], h0[ps], 1e-9, 1e-9,
                                     track=g.N - 1, log_cap=300)
        prop.prop_schedule(4.0, np.tile([0.1, 0.2], (len(ps), 1)))
        x2 = [prop.get_state(i) for i in range(len(ps))]
        prop.close()
        return pop, x1, st, np.asarray(log), x2

    every = list(range(P))
    pop, x1, st, log, x2 = run(every)
    assert st[0].rejected >= 1 and st[P // 2].attempts == 0
    for p in sorted({0, 1, P // 2, P - 1}):
        pop_, x1_, st_, log_, x2_ = run([p])
        assert np.array_equal(pop[p], pop_[0])
        assert np.array_equal(x1[p], x1_[0]) and np.array_equal(x2[p], x2_[0])
        assert (st[p].accepted, st[p].rejected, st[p].t, st[p].h) == (
            st_[0].accepted, st_[0].rejected, st_[0].t, st_[0].h)
        assert np.array_equal(log[p], log_[0])
    for graph, ms in ((False, 0), (True, -1)):
        _, y1, sy, _, y2 = run(every, graph, ms)
        assert [q.accepted for q in sy] == [q.accepted for q in st]
        assert np.abs(np.array(y1) - np.array(x1)).max() < 1e-12
        assert np.abs(np.array(y2) - np.array(x2)).max() < 1e-11


CHILD = """
import sys
import numpy as np
sys.path[:0] = [%r, %r]
import mpci
from mpci import synth
from test_gpu_rows import state
E, D = synth.system_arrays(%r, seed=9)
g = mpci.System(E, D)
p = mpci.Propagator(g)
p.set_state(state(g.N, 3))
p.prop_fixed(0.0, 0.1, np.full((1, 20), 0.02))
np.save(%r, p.get_state())
"""


@pytest.mark.parametrize("s", [[300, 257, 513], [1777, 2401]])
def test_second_process(mpci, tmp_path, s):
    """A second process is refused cooperative launches while this one holds
    them; its ordinary launch gives the same bits."""
    import os
    import subprocess
    import sys
    from mpci import synth
    E, D = synth.system_arrays(s, seed=9)
    g = mpci.System(E, D)
    p = mpci.Propagator(g)
    p.set_state(state(g.N, 3))
    p.prop_fixed(0.0, 0.1, np.full((1, 20), 0.02))
    out = str(tmp_path / "x.npy")
    code = CHILD % (os.path.dirname(os.path.dirname(mpci.__file__)),
                    os.path.dirname(os.path.abspath(__file__)), s, out)
    subprocess.run([sys.executable, "-c", code], check=True, timeout=100)
    assert np.array_equal(np.load(out), p.get_state())


def test_gives_up_and_goes_on(mpci):
    """A launch that may not wait leaves at once; the run goes on with one
    launch per stage from where it began, and so do later runs."""
    from mpci import synth
    E, D = synth.system_arrays([60, 75, 33], seed=3)
    g = mpci.System(E, D)
    x0 = state(g.N, 1)
    out = []
    for ms in (0, -1):
        prop = make(mpci, g, x0, True, "v")
        prop.set_wait_limit(ms)
        st, _ = prop.prop_adaptive(0.0, 5.0, 0.1, 1e-10, 1e-10)
        pop = prop.prop_fixed(0.0, 0.1, np.full((1, 30), 0.02))
        out.append((st[0].accepted, pop, prop.get_state()))
        prop.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_nan_state_does_not_wait(mpci):
    """A state that holds the exchange's marker bits (a signalling NaN no
    arithmetic produces) propagates like any other NaN."""
    from mpci import synth
    E, D = synth.system_arrays([20, 30], seed=4)
    g = mpci.System(E, D)
    x0 = state(g.N, 2)
    x0.view(np.uint64)[5] = 0x7FF4C0DEFACE0FF5
    prop = make(mpci, g, x0, True, "v")
    prop.prop_fixed(0.0, 0.1, np.full((1, 3), 0.02))
    assert np.isnan(prop.get_state()).all()


def test_concurrent_members(mpci):
    """Several one-pulse propagators at once, each with its own persistent
    launches, equal separate runs bit for bit."""
    from mpci import synth
    members = []
    for i, s in enumerate(([198] * 4, [300, 257, 513], [40, 30])):
        E, D = synth.system_arrays(s, seed=i)
        g = mpci.System(E, D)
        members.append((g, state(g.N, i)))
    ref, props = [], []
    for g, x0 in members:
        prop = make(mpci, g, x0, True, "v")
        prop.prop_adaptive(0.0, 9.0, 0.05, 1e-10, 1e-10)
        ref.append(prop.get_state())
        prop.set_state(x0)
        props.append(prop)
    n = len(props)
    mpci.multi_adaptive(props, [0.0] * n, [9.0] * n, [0.05] * n, 1e-10, 1e-10)
    for prop, r in zip(props, ref):
        assert np.array_equal(prop.get_state(), r)
