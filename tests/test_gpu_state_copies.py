"""States between the caller's memory and the batch layout: through a pinned
buffer holding all pulses, some of them at a time, or, past its size, none."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mpci():
    import mpci as m
    assert m.device_count() >= 1
    return m


@pytest.mark.parametrize("s,P", [([1, 2], 1), ([1, 2], 3), ([130, 127], 200),
                                 ([3000, 2900], 100), ([524300, 2], 1),
                                 ([524300, 2], 2)])
def test_states_and_rhs(mpci, s, P):
    """What goes in comes out bit for bit; the batch's RHS equals the pulses'
    own within rounding (1e-13) and leaves the states as they were."""
    from mpci import synth
    E, D = synth.system_arrays(s, seed=sum(s))
    g = mpci.System(E, D)
    rng = np.random.default_rng(P)
    x = rng.standard_normal((P, 2 * g.N))
    x /= np.linalg.norm(x, axis=1)[:, None]
    F = rng.standard_normal(P) * 0.05
    prop = mpci.Propagator(g, P=P)
    for p in range(P):
        prop.set_state(x[p], p)
    for p in range(P):
        assert np.array_equal(prop.get_state(p), x[p])
    k = prop.rhs(F, x).reshape(P, -1)
    for p in range(P):
        assert np.array_equal(prop.get_state(p), x[p])
    one = mpci.Propagator(g)
    for p in sorted({0, P // 2, P - 1}):
        assert np.abs(one.rhs(F[p], x[p]) - k[p]).max() < 1e-13
