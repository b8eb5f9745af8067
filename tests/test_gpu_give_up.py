"""The way back from a persistent launch that gives up after it has done work:
one workgroup leaves before a given attempt, the others stop waiting for it or,
in other groups of a batch, finish their pulses and write them.  The run has
to equal, bit for bit, the one that goes by launches of single stages from the
beginning: states, control records and logs are put back."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mpci():
    import mpci as m
    assert m.device_count() >= 1
    return m


def state(n, seed):
    x = np.random.default_rng(seed).standard_normal(2 * n)
    return x / np.linalg.norm(x)


# one pulse in rows and in tiles; batches of one group (slots), of several
# groups, and of groups that take a second set of pulses
@pytest.mark.parametrize("s,P,quits", [
    ([60, 75, 33], 1, (0, 1, 7)), ([300, 257, 513], 1, (3,)),
    ([1777, 2401], 1, (0, 3)), ([2400, 2500, 1300], 1, (2,)),
    ([2000, 2000], 2, (2,)), ([60, 72, 48], 100, (0, 2, 9)),
    ([950] + [2] * 20, 27, (0, 4, 12))])
def test_run_after_giving_up_midway(mpci, s, P, quits):
    from mpci import synth
    E, D = synth.system_arrays(s, seed=sum(s))
    g = mpci.System(E, D)
    F = 0.05 * np.sin(np.arange(13.0) + np.arange(P)[:, None])
    t1 = 3.0 + 0.3 * (np.arange(P) % 7)
    h0 = np.where(np.arange(P) == 0, 2.0, 0.1)

    def make(ms):
        prop = mpci.Propagator(g, P=P)
        for p in range(P):
            prop.set_state(state(g.N, 50 + p), p)
            prop.set_pulse(mpci.Pulse.sine(0.04 ** 2, 0.5 + 0.01 * p, 2), p)
        if ms is None:
            prop.set_graph(False)
        else:
            prop.set_wait_limit(ms)
        return prop

    def fixed(ms):
        prop = make(ms)
        pop = prop.prop_fixed(0.0, 0.1, F, track=g.N // 2)
        x = [prop.get_state(p) for p in range(P)]
        prop.close()
        return [pop, x]

    def adaptive(ms):
        prop = make(ms)
        st, log = prop.prop_adaptive(1.0, t1, h0, 1e-9, 1e-9, track=g.N - 1,
                                     log_cap=300)
        x = [prop.get_state(p) for p in range(P)]
        prop.close()
        return [[(q.accepted, q.rejected, q.attempts, q.t, q.h) for q in st],
                log, x]

    for run in (fixed, adaptive):
        ref, whole = run(None), run(0)
        # past the last attempt nothing is given up
        for a, b in zip(run(-2 - 1000), whole):
            assert np.array_equal(a, b)
        for n in quits:
            for a, b in zip(run(-2 - n), ref):
                assert np.array_equal(a, b), (run.__name__, n)
