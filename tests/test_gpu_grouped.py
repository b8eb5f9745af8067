"""Grouped launches (every member's attempt in the same launches) of batches
that run by launches on their own too, so that small members take part: each
member equals its own separate run bit for bit, members and pulses ending at
different times, whichever tile the group runs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 1e-10
SHAPES = [([24] * 9, 5, "v", 4), ([60, 72, 48], 3, "l", 2),
          ([300, 257, 310], 9, "v", 3)]


@pytest.fixture(scope="module")
def mpci():
    import mpci as m
    assert m.device_count() >= 1
    return m


@pytest.fixture(scope="module")
def members(mpci):
    from mpci import synth
    out = []
    for i, (s, P, gauge, most) in enumerate(SHAPES):
        E, D = synth.system_arrays(s, seed=70 + i)
        w, E0, cyc = synth.pulse_batch(P, seed=80 + i)
        cyc = np.minimum(cyc, 1 + np.arange(P) % most)
        out.append(dict(g=mpci.System(E, D, gauge=gauge), P=P, gauge=gauge,
                        t1=np.array([mpci.period(w[p], int(cyc[p]))
                                     for p in range(P)]),
                        pulses=[(E0[p] ** 2, w[p], int(cyc[p]))
                                for p in range(P)]))
    return out


def pin(prop, **want):
    for k in range(prop.gemm_candidates()):
        c = prop.set_gemm_candidate(k)
        if all(c[q] == v for q, v in want.items()):
            return
    raise AssertionError(want)


def fresh(mpci, m, tile, launches=True):
    from mpci import synth
    prop = mpci.Propagator(m["g"], P=m["P"])
    for p, (I, w, c) in enumerate(m["pulses"]):
        prop.set_state(synth.ground_state(m["g"].N), p)
        prop.set_pulse(mpci.Pulse.sine(I, w, c, m["gauge"]), p)
    if launches:
        prop.set_small_path(0)
    if tile:
        pin(prop, **tile)
    return prop


def check(mpci, ms, tiles, launches):
    make = lambda: [fresh(mpci, *a) for a in zip(ms, tiles, launches)]  # noqa
    props = make()
    st = mpci.multi_adaptive(props, [0.0] * len(ms), [m["t1"] for m in ms],
                             [0.05] * len(ms), TOL, TOL, grouped=True)
    assert len({q.attempts for x in st for q in x}) > 2  # uneven ends
    for m, prop, one, s in zip(ms, props, make(), st):
        s1, _ = one.prop_adaptive(0.0, m["t1"], 0.05, TOL, TOL)
        for p in range(m["P"]):
            assert (s[p].accepted, s[p].rejected, s[p].t, s[p].h) == (
                s1[p].accepted, s1[p].rejected, m["t1"][p], s1[p].h), p
            assert np.array_equal(prop.get_state(p), one.get_state(p)), p
        one.close()
        prop.close()


LDS = dict(kernel="k_gemm_lds")
PAIR = dict(kernel="k_gemm_pair", ksplit=1)


@pytest.mark.parametrize("lead", [
    {}, dict(LDS, wm=2, wn=2, fm=1, fn=1, ksplit=8),
    dict(LDS, wm=4, wn=2, fm=1, fn=1), dict(LDS, wm=4, wn=1, fm=1, fn=1),
    dict(LDS, wm=2, wn=2, fm=2, fn=1), dict(LDS, wm=4, wn=1, fm=2, fn=1),
    dict(LDS, wm=2, wn=1, fm=2, fn=2), dict(LDS, wm=4, wn=4, fm=2, fn=2),
    dict(kernel="k_gemm_db"), PAIR])
def test_grouped_launches_equal_separate_runs(mpci, members, lead):
    """The member with the most coupling work, the last, gives the tile."""
    check(mpci, members, [{}, dict(LDS, ksplit=2), lead], [True] * 3)


def test_pair_kernel_beside_grouped_panels(mpci, members):
    check(mpci, members, [PAIR, {}, dict(LDS, ksplit=4)], [True] * 3)


def test_persistent_members_beside_a_group(mpci, members):
    """The first two members run persistently, the third by launches."""
    check(mpci, members, [{}, {}, {}], [False, False, True])
    check(mpci, members, [{}, {}, {}], [False, True, True])


def test_persistent_members_in_one_launch(mpci, members):
    """Small batches that run persistently by themselves: grouped, their
    workgroups share one launch, with fewer groups and more pulses a group,
    and slots that take one pulse after another."""
    m = members
    check(mpci, [m[0], m[1]], [{}] * 2, [False] * 2)
    check(mpci, [m[0]] * 4 + [m[1], m[2]] + [m[0]] * 2, [{}] * 8, [False] * 8)
