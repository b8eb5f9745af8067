"""The engine's host code on a runtime of host memory (no GPU): what it
launches, keeps and gives back, and what it reads after a launch."""
import pytest

from host_runtime import host_runtime  # noqa: F401


@pytest.mark.parametrize("s,P", [([60, 75, 33], 1), ([1777, 2401], 1),
                                 ([60, 75, 33], 3)])
def test_old_give_up_does_not_undo_later_runs(host_runtime, s, P):  # noqa
    """A persistent launch that gave up leaves its flag on the device; with
    the persistent forms switched on again, runs that go by launches
    (eager, instrumented, the adjoint, grouped) keep what they computed."""
    host_runtime(f"""
    g, P = system({s}), {P}
    p = mpci.Propagator(g, P=P)
    x0 = np.arange(2.0 * g.N)
    for i in range(P):
        p.set_state(x0, i)
        p.set_pulse(mpci.Pulse.pwl(np.full(4, 0.01), 0.7, 100.0), i)
    F = np.full((P, 30), 0.02)
    n = 0

    def ran(k):
        global n
        n += k
        for i in range(P):
            assert np.array_equal(p.get_state(i), x0 + n), (n, i)

    def adaptive(run):
        st = run()
        assert all(q.accepted == 8 and q.t == 2.0 for q in st)
        ran(8)

    p.set_wait_limit(-1)
    p.prop_fixed(0.0, 0.1, F)
    ran(30)
    assert launches("k_apply") == 30  # it gave up
    p.set_wait_limit(0)
    p.set_small_path(-1)
    p.set_graph(False)
    p.prop_fixed(0.0, 0.1, F[:, :7])
    ran(7)
    one = lambda: p.prop_adaptive(0.0, 2.0, 0.25, 1e-9, 1e-9)[0]
    adaptive(one)
    p.set_graph(True)
    p.set_instrument(True)
    adaptive(one)
    p.set_instrument(False)
    W = np.ones(g.N)
    assert p.adjoint(0.0, 2.0, 0.25, W)[2].tolist() == [8] * P
    ran(8)
    if P > 1:
        p.set_graph(False)
        adaptive(lambda: mpci.multi_adaptive([p], [0.0], [2.0], [0.25], 1e-9,
                                             1e-9, grouped=True)[0])
        p.set_graph(True)
    rt.rt_clear()
    adaptive(one)
    assert launches("_run") == 1 and launches("k_apply") == 0
    """)


def test_row_kernel_reads_ahead_inside_its_lds(host_runtime):  # noqa: F811
    """k_rows_run reads the second copy of the neighbours' stage input one
    group of four 64-row chunks of 16-byte elements ahead while it works on
    chunks held in registers (16): its LDS has to reach there also where
    little else follows the copies."""
    host_runtime("""
    for s, P in (([1, 1], 1), ([198] * 4, 1), ([300] * 6, 1), ([64, 65], 1),
                 ([500, 500], 1), ([512, 512, 512], 1), ([513, 512, 512], 1),
                 ([1, 1], 3), ([198] * 4, 5), ([1025, 30, 1100], 1)):
        g = system(s)
        p = mpci.Propagator(g, P=P)
        p.prop_fixed(0.0, 0.1, np.full((P, 1), 0.02))
        assert launches("k_rows_run") == 1
        rt.rt_clear()
        ch = lambda n: (n + 63) // 64
        nch = [(ch(s[L - 1]) if L else 0) +
               (ch(s[L + 1]) if L + 1 < len(s) else 0) for L in range(len(s))]
        whole = [(n + 3) // 4 * 4 for n in nch]
        last = max(w + min(w, 16) + 4 for w in whole)
        assert rt.rt_lds() >= last * 64 * 16, (s, P, rt.rt_lds(), last)
    """)


REFUSED = """
def refused(f, code=-2):
    try:
        f()
    except mpci.MpciError as e:
        assert e.code == code, e
        return
    assert False, "accepted"
"""


def test_tables_grow_again_after_a_failed_allocation(host_runtime):  # noqa
    """A table that could not grow is allocated again by a smaller call."""
    host_runtime(REFUSED + """
g = system([60, 75, 33])
p = mpci.Propagator(g)
x0 = np.arange(2.0 * g.N)
p.set_state(x0)
huge = 1 << 18
rt.rt_fail_above(1 << 20)
refused(lambda: p.prop_fixed(0.0, 0.1, np.full((1, huge), 0.02)))
refused(lambda: p.prop_schedule(0.0, np.full((1, huge), 0.1)))
p.prop_fixed(0.0, 0.1, np.full((1, 5), 0.02))
p.prop_schedule(0.0, np.full((1, 6), 0.1))
assert np.array_equal(p.get_state(), x0 + 11)
""")


CANDIDATES = REFUSED + """
g = system([300, 280, 310])
p = mpci.Propagator(g, P=4)
held = {}
for k in range(p.gemm_candidates()):
    p.set_gemm_candidate(k)
    held[k] = rt.rt_live_bytes()
big, small = max(held, key=held.get), min(held, key=held.get)
mid = [k for k in held if held[small] < held[k] < held[big]][0]
split = (300 + 2 * 280 + 310) * 4 * 16   # partials of one K split
p.set_gemm_candidate(small)
rt.rt_fail_above(split)
refused(lambda: p.set_gemm_candidate(big))
"""


def test_tiles_after_one_that_did_not_fit(host_runtime):  # noqa: F811
    """After a candidate tile whose buffers did not fit, a smaller one gets
    its own (it was timed on no buffer at all)."""
    host_runtime(CANDIDATES + """
rt.rt_fail_above(1 << 40)
p.set_gemm_candidate(mid)
assert rt.rt_live_bytes() == held[mid]
p.prop_fixed(0.0, 0.1, np.full((4, 2), 0.02))
""")


def test_no_launch_without_coupling_buffers(host_runtime):  # noqa: F811
    """A propagator left without its coupling buffers by a tile that did not
    fit refuses to run until it has a tile again."""
    host_runtime(CANDIDATES + """
rt.rt_clear()
refused(lambda: p.prop_fixed(0.0, 0.1, np.full((4, 2), 0.02)), -3)
refused(lambda: p.rhs(0.02, np.ones(8 * g.N)), -3)
refused(lambda: mpci.multi_adaptive([p], [0.0], [2.0], [0.25], 1e-9, 1e-9,
                                    grouped=True), -3)
assert launches("k_gemm") == launches("7k_stage") == launches("k_apply") == 0
p.set_gemm_candidate(small)
p.prop_fixed(0.0, 0.1, np.full((4, 2), 0.02))
p.rhs(0.02, np.ones(8 * g.N))
""")


@pytest.mark.parametrize("grouped", [True, False])
def test_bad_argument_of_one_member_runs_none(host_runtime, grouped):  # noqa
    """An argument error of any member is found before a member runs, also
    where some run in persistent launches and the others grouped."""
    host_runtime(REFUSED + f"""
ps, xs = [], []
for i, s in enumerate(([60, 75, 33], [300, 280], [40, 41])):
    p = mpci.Propagator(system(s), P=2)
    if i == 1:
        p.set_small_path(0)
    x = np.arange(2.0 * sum(s))
    for k in range(2):
        p.set_state(x, k)
    ps.append(p)
    xs.append(x)
for bad in range(3):
    h = [0.25] * 3
    h[bad] = 0.0
    refused(lambda: mpci.multi_adaptive(ps, [0.0] * 3, [2.0] * 3, h, 1e-9,
                                        1e-9, grouped={grouped}), -1)
    for p, x in zip(ps, xs):
        assert np.array_equal(p.get_state(0), x)
mpci.multi_adaptive(ps, [0.0] * 3, [2.0] * 3, [0.25] * 3, 1e-9, 1e-9,
                    grouped={grouped})
for p, x in zip(ps, xs):
    assert np.array_equal(p.get_state(1), x + 8)
""")


def test_pinned_tile_stays(host_runtime):  # noqa: F811
    """A pinned tile is what a batch runs, also after the small-system path
    has been chosen anew."""
    host_runtime("""
    g = system([60, 75, 33])
    p = mpci.Propagator(g, P=5)
    F = np.full((5, 4), 0.02)
    p.prop_fixed(0.0, 0.1, F)
    assert launches("k_rows_run") == 1
    p.set_gemm_candidate(2)
    for mode in (-1, 1, 0):
        p.set_small_path(mode)
        rt.rt_clear()
        p.prop_fixed(0.0, 0.1, F)
        assert launches("k_rows_run") == 0 and launches("k_gemm") == 4 * 13
    """)


@pytest.mark.parametrize("s,P,kernel", [([1201, 1333, 997], 1, "k_relayout_r"),
                                        ([300, 280, 310], 40, "k_gemm_db")])
def test_propagators_created_in_threads(host_runtime, s, P, kernel):  # noqa
    """Several threads create propagators of one system: its row store is
    built once, and its tile searched once, as one after the other."""
    host_runtime(f"""
    import threading
    counts = []
    for n in (1, 6):
        g = system({s})
        rt.rt_clear()
        rt.rt_alloc_us(2000)
        ps = [None] * n

        def make(i):
            ps[i] = mpci.Propagator(g, P={P})

        ts = [threading.Thread(target=make, args=(i,)) for i in range(n)]
        [t.start() for t in ts]
        [t.join() for t in ts]
        counts.append(launches("{kernel}"))
        rt.rt_alloc_us(0)
        [p.close() for p in ps]
        g.close()
        assert rt.rt_live() == 0
    assert counts[0] == counts[1] > 0, counts
    """)


@pytest.mark.parametrize("s,P,first", [
    ([198] * 4, 1, "row store"), ([1201, 1333, 997], 1, "row store"),
    ([1201, 1333, 997], 1, "exchange"), ([1777, 2401], 1, "exchange"),
    ([300, 280, 310], 5, "row store"), ([300, 280, 310], 5, "exchange")])
def test_persistent_form_without_room(host_runtime, s, P, first):  # noqa
    """Where the row store or the exchange buffers do not fit, a propagator
    is created all the same, runs by launches and holds nothing of the form;
    it has the form when it is asked for again and there is room."""
    n16 = sum(-(-n // 16) for n in s)
    ch = [-(-n // 64) for n in s]
    store = 4 * 64 * 8 * sum(
        -(-n // 4) * (sum(ch[max(L - 1, 0):L]) + sum(ch[L + 1:L + 2]))
        for L, n in enumerate(s))
    groups = min(P, max(256 // n16, 1))
    copies = 3 if n16 > 256 else 4 * groups * -(-P // groups)
    size = store if first == "row store" else 16 * sum(s) * copies
    host_runtime(f"""
    s, P = {s}, {P}
    F, x0 = np.full((P, 2), 0.02), np.arange(2.0 * sum(s))

    def run(p, persistent):
        p.set_state(x0)
        rt.rt_clear()
        p.prop_fixed(0.0, 0.1, F)
        assert np.array_equal(p.get_state(), x0 + 2)
        assert launches("_run") == persistent
        assert launches("k_apply") == (0 if persistent else 2)
        return rt.rt_live_bytes()

    rt.rt_fail_at.argtypes = [ctypes.c_size_t] * 2
    g = system(s)
    p = mpci.Propagator(g, P=P)
    held = run(p, True)
    p.close(), g.close()
    rt.rt_fail_at({size}, {size})
    g = system(s)
    p = mpci.Propagator(g, P=P)
    assert run(p, False) <= held - {size if n16 > 256 else store}
    p.rhs(0.02, np.ones(2 * g.N * P))
    rt.rt_fail_at(1, 0)
    p.set_small_path(-1)
    assert run(p, True) == held
    p.close(), g.close()
    assert rt.rt_live() == 0
    """)


def test_persistent_launches_are_bounded(host_runtime):  # noqa: F811
    """A persistent launch holds the device, so it takes a stated time at
    most: by the time of its attempts 100 ms alone, 20 ms beside others (a
    row attempt at least 30 us and a pass, a tile attempt at least 13 sweeps
    of the dipoles at 7 TB/s)."""
    host_runtime("""
    def run(members, together):
        ps = []
        for s, P in members:
            p = mpci.Propagator(system(s), P=P)
            p.set_state(np.zeros(2 * sum(s)))
            ps.append(p)
        rt.rt_clear()
        for q in [ps] if together else [[p] for p in ps]:
            n = len(q)
            st = mpci.multi_adaptive(q, [0.0] * n, [1024.0] * n, [0.25] * n,
                                     1e-9, 1e-9)
            assert all(x[0].accepted == 4096 for x in st)
        a = attempts()
        for p in ps:
            assert np.array_equal(p.get_state(), np.full(2 * p.sys.N, 4096.0))
        assert sum(a) >= 4096 * len(members)
        return a

    small, tiles, batch = ([198] * 4, 1), ([1500] * 4, 1), ([60] * 8, 5)
    one = 13 * 8 * 3 * 1500 ** 2 / 7e6  # us
    assert max(run([small], False)) * 30.0 <= 100e3
    assert max(run([tiles], False)) * one <= 100e3
    a = run([small, batch], True)
    assert max(a) * 30.0 <= 20e3 and min(a) >= 16
    a = run([tiles, small], True)
    assert min(a) * one <= 20e3 and min(a) >= 16
    p = mpci.Propagator(system([1500] * 4))
    rt.rt_clear()
    p.prop_fixed(0.0, 0.1, np.full((1, 4500), 0.02))
    assert max(attempts()) * one <= 100e3
    """)


@pytest.mark.parametrize("s,P", [([60, 75, 33], 1), ([30, 20], 3)])
@pytest.mark.parametrize("steps,K", [(1000, 32), (1000, 8), (992, 32),
                                     (20, 32), (32, 32), (33, 32), (5, 1)])
def test_adjoint_keeps_little_more_than_it_uses(host_runtime, s, P, steps, K):  # noqa
    """The adjoint's forward pass keeps the stage inputs of its last segment,
    and of few steps besides: the first segment's (a short run has no other)
    and those of the last four segments.  The last segment is not propagated
    again."""
    host_runtime(f"""
    g, P, steps, K = system({s}), {P}, {steps}, {K}
    p = mpci.Propagator(g, P=P)
    for i in range(P):
        p.set_state(np.arange(2.0 * g.N), i)
        p.set_pulse(mpci.Pulse.pwl(np.full(4, 0.01), 0.7, 2000.0), i)
    nst, st = p.adjoint(0.0, 0.25 * steps, 0.25, np.ones(g.N),
                        ckpt_every=K)[2::2]
    assert nst.tolist() == [steps] * P
    again = (steps - 1) // K * K   # all but the last segment
    kept = rt.rt_stored() - 13 * again
    assert kept % 13 == 0 and steps - again <= kept // 13 <= 6 * K, kept
    if steps <= K:
        assert kept == 13 * steps
    """)


def test_one_slow_launch_does_not_drop_a_tile(host_runtime):  # noqa: F811
    """The tile search leaves a candidate after a slow evaluation only when a
    second one is slow as well."""
    host_runtime("""
    g = system([300, 280, 310])
    # k_gemm_lds of 4 x 1 waves and 2 x 1 blocks: the fastest, but slow once
    rt.rt_cost(b"k_gemm", 100.0, 100.0, 0)
    rt.rt_cost(b"k_gemm_ldsILi4ELi1ELi2ELi1E", 1.0, 1e5, 2)
    c = mpci.Propagator(g, P=40).gemm_config()
    assert (c["kernel"], c["wm"], c["wn"], c["fm"], c["fn"]) == (
        "k_gemm_lds", 4, 1, 2, 1), c
    assert c["ms"] < 0.02
    # always slow ones are left after two looks
    rt.rt_cost(b"k_gemm_pair", 1e5, 1e5, 0)
    rt.rt_clear()
    g = system([300, 280, 310])
    assert mpci.Propagator(g, P=40).gemm_config() == c
    assert launches("k_gemm_pair") == 2 * 3
    """)


@pytest.mark.parametrize("wm,wn,fm,fn", [(2, 2, 1, 1), (4, 2, 1, 1),
                                         (2, 2, 2, 1), (4, 1, 1, 1),
                                         (4, 1, 2, 1), (4, 2, 2, 2)])
def test_group_runs_the_tile_of_its_largest_member(host_runtime, wm, wn, fm,  # noqa
                                                   fn):
    """The grouped launches take the tile that was timed for the member with
    the most coupling work, its blocks a wave as well as its waves."""
    host_runtime(f"""
    want = dict(kernel="k_gemm_lds", wm={wm}, wn={wn}, fm={fm}, fn={fn})
    ps = [mpci.Propagator(system(s), P=20) for s in ([300, 280], [70, 60, 50])]
    for k in range(ps[0].gemm_candidates()):
        c = ps[0].set_gemm_candidate(k)
        if all(c[q] == v for q, v in want.items()):
            break
    else:
        assert False, "no such candidate"
    ps[1].set_small_path(0)
    rt.rt_clear()
    mpci.multi_adaptive(ps, [0.0] * 2, [2.0] * 2, [0.25] * 2, 1e-9, 1e-9,
                        grouped=True)
    name = "k_gemm_lds_gILi{wm}ELi{wn}ELi{fm}ELi{fn}E"
    assert launches(name) == launches("k_gemm") >= 8 * 13
    assert launches("k_apply_g") >= 8 and launches("_run") == 0
    """)


def test_every_candidate_tile_is_launched(host_runtime):  # noqa: F811
    host_runtime("""
    p = mpci.Propagator(system([300, 280]), P=3)
    for k in range(p.gemm_candidates()):
        c = p.set_gemm_candidate(k)
        rt.rt_clear()
        p.prop_fixed(0.0, 0.1, np.full((3, 1), 0.02))
        assert launches(c["kernel"]) == launches("k_gemm") == 13, c
    """)


def test_grouped_row_members_share_launches(host_runtime):  # noqa: F811
    """Grouped members in the row form run in launches for all of them; one
    that gives up goes on by launches of single stages; too many rows for the
    device together run one after the other."""
    host_runtime("""
    def run(shapes, quits=()):
        ps = []
        for i, (s, P) in enumerate(shapes):
            p = mpci.Propagator(system(s), P=P)
            for k in range(P):
                p.set_state(np.arange(2.0 * sum(s)), k)
            if i in quits:
                p.set_wait_limit(-1)
            ps.append(p)
        n = len(ps)
        t1 = [2.0 + i + np.arange(p.P) for i, p in enumerate(ps)]
        rt.rt_clear()
        before = rt.rt_live()
        st = mpci.multi_adaptive(ps, [0.0] * n, t1, [0.25] * n, 1e-9, 1e-9,
                                 grouped=True)
        assert rt.rt_live() <= before
        for i, p in enumerate(ps):
            for k in range(p.P):
                steps = int(t1[i][k] / 0.25)
                assert st[i][k].accepted == steps and st[i][k].t == t1[i][k]
                assert np.array_equal(p.get_state(k),
                                      np.arange(2.0 * p.sys.N) + steps)
        return launches("k_rows_run"), launches("k_apply")

    assert run([([60] * 8, 5)] * 8) == (1, 0)
    assert run([([60] * 8, 5), ([40, 30], 3), ([198] * 4, 9)]) == (1, 0)
    n, apply = run([([60] * 8, 5), ([40, 30], 3), ([198] * 4, 2)], [1])
    assert n == 1 and 20 <= apply < 40     # (plus what was planned past the end)
    assert run([([300] * 6, 5)] * 3) == (3, 0)
    # no gain (two pulses a group each), and a third in grouped launches
    assert run([([60] * 8, 5)] * 2 + [([300, 280], 200)])[0] == 2
    """)


@pytest.mark.parametrize("s,P", [([60, 75, 33], 1), ([1777, 2401], 1),
                                 ([60, 75, 33], 3)])
def test_work_of_a_launch_that_gave_up_is_undone(host_runtime, s, P):  # noqa
    """States, control records and log entries written before a launch gave
    up are put back; the run counts every step once."""
    host_runtime(f"""
    g, P = system({s}), {P}
    for n in (0, 3, 8):
        rt.rt_abort_after(n)
        p = mpci.Propagator(g, P=P)
        x0 = np.arange(2.0 * g.N)
        for i in range(P):
            p.set_state(x0 + i, i)
        rt.rt_clear()
        st, log = p.prop_adaptive(0.0, 2.0, 0.25, 1e-9, 1e-9, log_cap=20)
        assert launches("_run") == 1 and launches("k_apply") >= 8
        for i in range(P):
            assert (st[i].accepted, st[i].attempts, st[i].t) == (8, 8, 2.0)
            assert np.array_equal(p.get_state(i), x0 + i + 8)
            assert log[i, :8, 0].tolist() == [0.25 * (k + 1) for k in range(8)]
        p.close()
    """)


def test_tile_search_leaves_out_what_does_not_fit(host_runtime):  # noqa: F811
    """Creating a batch needs room for the tile it runs: candidates with finer
    K splits, whose partials do not fit, are left out."""
    split = (300 + 2 * 280 + 310) * 40 * 16   # partials of one K split
    host_runtime(REFUSED + f"""
rt.rt_cost(b"k_gemm", 100.0, 100.0, 0)
rt.rt_fail_multiples.argtypes = [ctypes.c_size_t] * 2
for most in (8, 4, 2, 1):
    rt.rt_fail_multiples({split}, most)
    g = system([300, 280, 310])
    p = mpci.Propagator(g, P=40)
    assert p.gemm_config()["ksplit"] <= most
    p.prop_fixed(0.0, 0.1, np.full((40, 2), 0.02))
    p.close(), g.close()
    assert rt.rt_live() == 0
rt.rt_fail_multiples({split}, 0)   # no tile fits
g = system([300, 280, 310])
refused(lambda: mpci.Propagator(g, P=40))
""")
