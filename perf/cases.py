"""Timed cases of the propagation library: what a program asks of it, from one
right-hand side on a small hydrogen basis to batches of pulses on the large
helium basis, forward and backward, through the Python mirror of the C ABI.

Systems are synthetic, in the shapes this repository uses: the block sizes of
tests/golden/*.yaml, those of bench.py (He 4 x 4000, H 21 x 998, H 4 x 198)
and odd ones between.  Energies are uniform and sorted per block, dipoles
N(0, 1/s_{L+1}) as mpci.synth draws them; the state is that of a run under
way (mostly the ground state, the rest spread over the spectrum), the field
that of the middle of a pulse.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "mp-citdse_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "mp-citdse_amd"))

DT = 0.1             # dt of tests/golden/*.yaml
THRESHOLD = -2.0     # one-electron threshold of the yield weights (a.u.)


def listed():
    return [
        # the smallest call: one RHS on the H basis, host arrays in and out
        # (an integrator of the caller's own)
        dict(name="rhs_h4x198", kind="rhs", blocks="198x4", P=1, gauge="v",
             e_lo=-0.5),
        # the same operator applied to device buffers, the large He basis
        dict(name="rhs_device_he4x4000", kind="rhs_device", blocks="4000x4",
             P=1, gauge="v", e_lo=-2.9),
        # tdse -e 1: one tenth of the pulse between two coefficient files
        dict(name="fixed_h4x198", kind="fixed", blocks="198x4", P=1,
             gauge="v", e_lo=-0.5, shape="sine", w=0.5, E0=0.05, cycles=10,
             steps=125),
        # the same with the blocks of H_test.yaml
        dict(name="fixed_h6x300", kind="fixed", blocks="300x6", P=1,
             gauge="v", e_lo=-0.5, shape="sine", w=0.3124, E0=0.0169,
             cycles=12, steps=120),
        # odd middle-sized blocks, length gauge, gaussian pulse, adaptive
        dict(name="adaptive_odd", kind="adaptive", blocks="1201,1333,997",
             P=1, gauge="l", e_lo=-2.9, shape="gaussian", w=0.7, E0=0.03,
             cycles=10, span=2.0, tol=1e-10),
        # tdse -e 2 with the blocks of He_test.yaml, reference mode
        dict(name="fixed_hetest", kind="fixed",
             blocks="3030,2799,2808,2808", P=1, gauge="v", e_lo=-2.9,
             shape="sine", w=0.7, E0=0.03, cycles=10, steps=40),
        # the large He basis, one pulse, adaptive at 1e-10, observables after
        dict(name="adaptive_he4x4000", kind="adaptive", blocks="4000x4", P=1,
             gauge="v", e_lo=-2.9, shape="sine", w=0.7, E0=0.03, cycles=10,
             span=2.0, tol=1e-10),
        # a small odd batch on a small basis
        dict(name="batch5_h6x300", kind="fixed", blocks="300x6", P=5,
             gauge="l", e_lo=-0.5, shape="sine", w=0.5, E0=0.03, cycles=8,
             steps=40),
        # many narrow blocks, a batch of 32 pulses
        dict(name="batch32_h21x998", kind="adaptive", blocks="998x21", P=32,
             gauge="v", e_lo=-0.5, shape="sine", w=0.7, E0=0.03, cycles=10,
             span=1.0, tol=1e-10),
        # 64 pulses on the large He basis
        dict(name="batch64_he4x4000", kind="adaptive", blocks="4000x4", P=64,
             gauge="v", e_lo=-2.9, shape="sine", w=0.7, E0=0.03, cycles=10,
             span=1.0, tol=1e-10),
        # pulse shaping: gradients of 16 envelopes on the large He basis
        dict(name="adjoint16_he4x4000", kind="adjoint", blocks="4000x4", P=16,
             gauge="v", e_lo=-2.9, w=0.7, E0=0.04, samples=4, span=2.0,
             tol=1e-6),
        # two instances at once: 32 pulses on H, 32 on He
        dict(name="multi32_h21x998_he4x4000", kind="multi", blocks="998x21",
             P=32, blocks2="4000x4", P2=32, gauge="v", e_lo=-0.5,
             shape="sine", w=0.7, E0=0.03, cycles=10, span=0.6, tol=1e-10),
    ]


def sizes(text):
    if "x" in text:
        n, k = text.split("x")
        return [int(n)] * int(k)
    return [int(n) for n in text.split(",")]


def elements(text):
    s = sizes(text)
    return sum(a * b for a, b in zip(s, s[1:]))


def draw(rng):
    kind = rng.choice(["rhs", "rhs_device", "fixed", "fixed", "adaptive",
                       "adaptive", "adjoint", "multi"])
    single = kind == "rhs_device" or (kind in ("rhs", "fixed", "adaptive") and
                                      rng.random() < 0.5)

    def pulses(most):
        return int(round(math.exp(rng.uniform(math.log(2), math.log(most)))))

    def blocks(most):
        nb = rng.randint(2, 8)
        top = min(4000, int(math.sqrt(most / (nb - 1))))
        n = math.exp(rng.uniform(math.log(60), math.log(max(top, 61))))
        s = [max(1, min(4000, int(n * rng.uniform(0.8, 1.1))))
             for _ in range(nb)]
        return ",".join(str(x) for x in s)

    P = 1 if single else pulses(16 if kind == "adjoint" else 64)
    c = dict(kind=kind, blocks=blocks(40e6), P=P, gauge=rng.choice("vl"),
             e_lo=rng.choice([-0.5, -2.9]))
    if kind in ("rhs", "rhs_device"):
        return c
    c.update(w=round(rng.uniform(0.5, 1.0), 3),
             E0=round(math.exp(rng.uniform(math.log(0.005), math.log(0.05))),
                      4))
    if kind == "adjoint":
        c.update(samples=rng.randint(2, 4), span=2.0, tol=1e-6)
        return c
    c.update(shape=rng.choice(["sine", "gaussian"]), cycles=rng.randint(4, 20))
    if kind == "fixed":
        c["steps"] = rng.randint(11, 120 if P == 1 else 40)
        while 8 * 13 * P * elements(c["blocks"]) * c["steps"] > 3e12:
            c["steps"] = (c["steps"] + 1) // 2
    else:
        c.update(span=1.0 if kind == "adaptive" else 0.6, tol=1e-10)
        if kind == "multi":
            c.update(P=pulses(16), blocks2=blocks(10e6), P2=pulses(16))
    return c


# ---- inputs from the seed ------------------------------------------------
def generator(seed, k):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 16 + k)
    return g


def operator(text, e_lo, seed, k=0):
    """Energies (host) and dipole blocks (device) of one system."""
    s = sizes(text)
    g = generator(seed, k)
    E = [torch.sort(torch.rand(n, dtype=torch.float64, device="cuda",
                               generator=g) * (5.0 - e_lo) + e_lo)[0]
         for n in s]
    D = [torch.randn(a, b, dtype=torch.float64, device="cuda", generator=g)
         / math.sqrt(b) for a, b in zip(s, s[1:])]
    return E, D


def states(E, P, seed, k=1):
    """P states of a run under way, (N, P) complex on the device: the ground
    state and a tail that falls off over the spectrum, of norm 1."""
    e = torch.cat(E)
    g = generator(seed, k)
    x = torch.randn(len(e), P, 2, dtype=torch.float64, device="cuda",
                    generator=g)
    x = x * torch.exp(-2.0 * (e - e.min()))[:, None, None]
    x = 0.4 * x / torch.sqrt((x * x).sum(dim=(0, 2), keepdim=True))
    x[0, :, 0] += 0.9
    x = x / torch.sqrt((x * x).sum(dim=(0, 2), keepdim=True))
    return torch.view_as_complex(x.contiguous())


class Field:
    """One laser pulse: its closed form here, its parameters for the library."""

    def __init__(self, c, p):
        self.gauge, self.shape = c["gauge"], c["shape"]
        self.w = c["w"] * (1.0 + 0.01 * p)
        self.E0, self.cycles = c["E0"] * (1.0 + 0.02 * (p % 7)), c["cycles"]
        self.tau = self.cycles * 2.0 * math.pi / self.w
        self.amp = self.E0 / self.w if self.gauge == "v" else self.E0

    def __call__(self, t):
        if not 0.0 <= t <= self.tau:
            return 0.0
        if self.shape == "sine":
            env = math.sin(self.w / (2.0 * self.cycles) * t) ** 2
        else:
            a = (0.5 * (2.0 * math.pi / self.w) * (2 + self.cycles // 10)
                 / 0.58870501125773734549)
            env = math.exp(-((t - 0.5 * self.tau) / a) ** 2)
        return self.amp * env * math.sin(self.w * t)

    def pulse(self, mpci):
        if self.shape == "sine":
            return mpci.Pulse.sine(self.E0 ** 2, self.w, self.cycles,
                                   gauge=self.gauge)
        return mpci.Pulse.gauss(self.E0 ** 2, self.w, self.tau, self.cycles,
                                gauge=self.gauge)


class Envelope:
    """A piecewise-linear envelope over [0, T] with carrier w."""

    def __init__(self, env, w, T, gauge):
        self.env, self.w, self.T = env, w, T
        self.scale = 1.0 / w if gauge == "v" else 1.0

    def __call__(self, t):  # t: (P,) times, env: (P, K) with gradients
        K = self.env.shape[1]
        u = t / (self.T / (K - 1))
        k = u.floor().long().clamp(0, K - 2)
        f = u - k
        r = torch.arange(len(t), device=t.device)
        en = (1.0 - f) * self.env[r, k] + f * self.env[r, k + 1]
        return self.scale * en * torch.sin(self.w * t)


def start_time(c, f):
    """Where in the pulse the timed part begins: near its peak."""
    return math.floor(0.45 * f.tau / DT) * DT


def interleaved(x):
    """(N, P) complex -> P host vectors of 2N doubles."""
    return [np.ascontiguousarray(v) for v in
            torch.view_as_real(x.t().contiguous()).reshape(x.shape[1], -1)
            .cpu().numpy()]


def envelopes(c, seed):
    return c["E0"] * torch.rand(c["P"], c["samples"], dtype=torch.float64,
                                device="cuda", generator=generator(seed, 3))


def fields_fixed(c, seed):
    """(P, steps) frozen fields F(t + dt), t accumulated as the loop does."""
    F = np.empty((c["P"], c["steps"]))
    for p in range(c["P"]):
        f = Field(c, p)
        t = start_time(c, f)
        for k in range(c["steps"]):
            F[p, k] = f(t + DT)
            t += DT
    return F


def rhs_fields(c, seed):
    return np.random.default_rng(int(seed)).uniform(-0.05, 0.05, c["P"])


class State:
    pass


def system(mpci, st, c, seed, k, blocks, P):
    E, D = operator(blocks, c["e_lo"], seed, k)
    sysg = mpci.System([e.cpu().numpy() for e in E],
                       [d.cpu().numpy() for d in D], gauge=c["gauge"])
    del D
    prop = mpci.Propagator(sysg, P=P)
    x0 = interleaved(states(E, P, seed, k + 1))
    st.keep += [sysg]
    return sysg, prop, x0


def prepare(case, seed):
    import mpci
    st = State()
    st.kind, st.keep = case["kind"], []
    c = case
    if st.kind == "rhs_device":
        from mpci import _lib
        E, D = operator(c["blocks"], c["e_lo"], seed)
        st.sys = mpci.System([e.cpu().numpy() for e in E],
                             [d.cpu().numpy() for d in D], gauge=c["gauge"])
        st.F = float(rhs_fields(c, seed)[0])
        st.x = torch.view_as_real(states(E, 1, seed)).reshape(-1).contiguous()
        st.out = torch.empty_like(st.x)
        st.call, st.check = _lib.tdse_lib().mpci_system_rhs_noalloc, _lib.check
        return st
    st.sys, st.prop, st.x0 = system(mpci, st, c, seed, 0, c["blocks"], c["P"])
    if st.kind == "rhs":
        st.F, st.x = rhs_fields(c, seed), np.concatenate(st.x0)
    elif st.kind == "fixed":
        st.F = fields_fixed(c, seed)
        st.t0 = start_time(c, Field(c, 0))
    elif st.kind == "adjoint":
        st.T, st.tol = c["span"], c["tol"]
        st.W = np.zeros(st.sys.N)
        st.W[:sizes(c["blocks"])[0]] = 1.0
        env = envelopes(c, seed).cpu().numpy()
        st.pulses = [mpci.Pulse.pwl(e, c["w"], st.T, gauge=c["gauge"])
                     for e in env]
    else:
        st.tol, st.members = c["tol"], []
        parts = [(st.sys, st.prop, st.x0)]
        if st.kind == "multi":
            parts.append(system(mpci, st, c, seed, 4, c["blocks2"], c["P2"]))
        for _, prop, x0 in parts:
            fs = [Field(c, p) for p in range(prop.P)]
            t0 = np.array([start_time(c, f) for f in fs])
            for p, f in enumerate(fs):
                prop.set_pulse(f.pulse(mpci), p)
            st.members.append((prop, x0, t0, t0 + c["span"]))
        st.multi = mpci.multi_adaptive
    return st


def run(st):
    """One pass: the states go in from host memory, the propagation runs, the
    states and what a program reads beside them come out."""
    if st.kind == "rhs_device":
        st.check(st.call(st.sys.h, st.F, st.x.data_ptr(), st.out.data_ptr(),
                         torch.cuda.current_stream().cuda_stream))
        return st.out
    prop = st.prop
    if st.kind == "rhs":
        return prop.rhs(st.F, st.x)
    if st.kind == "fixed":
        for p, x in enumerate(st.x0):
            prop.set_state(x, p)
        pop = prop.prop_fixed(st.t0, DT, st.F, track=0)
        return {"pop": pop, "x": np.stack([prop.get_state(p)
                                           for p in range(prop.P)])}
    if st.kind == "adjoint":
        for p, x in enumerate(st.x0):
            prop.set_state(x, p)
            prop.set_pulse(st.pulses[p], p)
        J, grad, nst, _, _ = prop.adjoint(0.0, st.T, DT, st.W, atol=st.tol,
                                          rtol=st.tol)
        return {"J": J, "grad": grad, "steps": nst}
    for prop, x0, _, _ in st.members:
        for p, x in enumerate(x0):
            prop.set_state(x, p)
    if st.kind == "multi":
        m = st.members
        stats = st.multi([x[0] for x in m], [x[2] for x in m],
                         [x[3] for x in m], [DT] * len(m), st.tol, st.tol)
    else:
        prop, _, t0, t1 = st.members[0]
        stats = [prop.prop_adaptive(t0, t1, DT, st.tol, st.tol)[0]]
    return [{"accepted": np.array([s.accepted for s in sm]),
             "rejected": np.array([s.rejected for s in sm]),
             "obs": prop.observables(2, THRESHOLD),
             "x": np.stack([prop.get_state(p) for p in range(prop.P)])}
            for sm, (prop, _, _, _) in zip(stats, st.members)]


def work(case):
    """Each RHS evaluation reads every dipole element and the state once and
    writes the derivative once; 8 P S flops (both products, Re and Im).  An
    adaptive step is taken to be DT long, a step of the adjoint a forward and
    a backward evaluation of its 13 stages."""
    c = case
    n = {"rhs": 1, "rhs_device": 1, "fixed": 13 * c.get("steps", 0)}.get(
        c["kind"])
    if n is None:
        n = 13 * max(1, round(c["span"] / DT))
        if c["kind"] == "adjoint":
            n = 2 * 13 * max(1, round(c["span"] / DT / 2))
    parts = [(c["blocks"], c["P"])]
    if c["kind"] == "multi":
        parts.append((c["blocks2"], c["P2"]))
    w = {"bytes": 0.0, "flops": 0.0}
    for blocks, P in parts:
        S, N = elements(blocks), sum(sizes(blocks))
        w["bytes"] += n * (8.0 * S + 32.0 * N * P)
        w["flops"] += n * 8.0 * P * S
    return w


# ---- the same in plain torch, 64 bits ------------------------------------
# Fehlberg's 7(8) pair (NASA TR R-287)
A = [[], [2 / 27], [1 / 36, 1 / 12], [1 / 24, 0, 1 / 8],
     [5 / 12, 0, -25 / 16, 25 / 16], [1 / 20, 0, 0, 1 / 4, 1 / 5],
     [-25 / 108, 0, 0, 125 / 108, -65 / 27, 125 / 54],
     [31 / 300, 0, 0, 0, 61 / 225, -2 / 9, 13 / 900],
     [2, 0, 0, -53 / 6, 704 / 45, -107 / 9, 67 / 90, 3],
     [-91 / 108, 0, 0, 23 / 108, -976 / 135, 311 / 54, -19 / 60, 17 / 6,
      -1 / 12],
     [2383 / 4100, 0, 0, -341 / 164, 4496 / 1025, -301 / 82, 2133 / 4100,
      45 / 82, 45 / 164, 18 / 41],
     [3 / 205, 0, 0, 0, 0, -6 / 41, -3 / 205, -3 / 41, 3 / 41, 6 / 41, 0],
     [-1777 / 4100, 0, 0, -341 / 164, 4496 / 1025, -289 / 82, 2193 / 4100,
      51 / 82, 33 / 164, 12 / 41, 0, 1]]
B = [0, 0, 0, 0, 0, 34 / 105, 9 / 35, 9 / 35, 9 / 280, 9 / 280, 0, 41 / 840,
     41 / 840]
DB = [-41 / 840, 0, 0, 0, 0, 0, 0, 0, 0, 0, -41 / 840, 41 / 840, 41 / 840]
C = [0, 2 / 27, 1 / 9, 1 / 6, 5 / 12, 1 / 2, 5 / 6, 1 / 6, 2 / 3, 1 / 3, 1, 0,
     1]


def derivative(E, D, gauge, x, F):
    """dx/dt for x (N, P) complex at fields F (P,)."""
    def times(m, v):
        r = torch.view_as_real(v).reshape(v.shape[0], -1)
        return torch.view_as_complex((m @ r).reshape(m.shape[0], -1, 2)
                                     .contiguous())
    xs = list(torch.split(x, [len(e) for e in E]))
    k = []
    for L, e in enumerate(E):
        up = times(D[L - 1].t(), xs[L - 1].contiguous()) if L > 0 else 0.0
        dn = (times(D[L], xs[L + 1].contiguous()) if L + 1 < len(E) else 0.0)
        if gauge == "v":
            k.append(-1j * e[:, None] * xs[L] + F * (up - dn))
        else:
            k.append(-1j * (e[:, None] * xs[L] + F * (up + dn)))
    return torch.cat(k)


def attempt(f, x, t, h, field):
    """Candidate state, error estimate and first derivative of one step; t, h
    (P,), field(t) (P,)."""
    k = []
    for s in range(13):
        xs = x
        for j in range(s):
            if A[s][j]:
                xs = xs + (h * A[s][j]) * k[j]
        k.append(f(xs, field(t + C[s] * h)))
    y, err = x, 0.0
    for j in range(13):
        if B[j]:
            y = y + (h * B[j]) * k[j]
        if DB[j]:
            err = err + (h * DB[j]) * k[j]
    return y, err, k[0]


def normalised(y):
    return y / torch.sqrt((y.real ** 2 + y.imag ** 2).sum(0))


def controlled(f, x, t0, t1, tol, field):
    """Adaptive run; returns the state and the per-pulse accepted counts."""
    t, h = t0.clone(), torch.full_like(t0, DT)
    acc, rej = torch.zeros_like(t0), torch.zeros_like(t0)
    live = t < t1
    while bool(live.any()):
        last = t + h >= t1
        hc = torch.where(live, torch.where(last, t1 - t, h),
                         torch.zeros_like(h))
        with torch.no_grad():
            y, err, k1 = attempt(f, x, t, hc, field)
            e = torch.zeros_like(t)
            for er, xr, kr in ((err.real, x.real, k1.real),
                               (err.imag, x.imag, k1.imag)):
                r = er.abs() / (tol + tol * (xr.abs() + hc * kr.abs()))
                e = torch.maximum(e, r.amax(0))
        ok = (e <= 1.0) & live
        if torch.is_grad_enabled():
            y, _, _ = attempt(f, x, t, hc, field)
        x = torch.where(ok, normalised(y), x)
        bad = live & ~ok
        acc, rej = acc + ok, rej + bad
        t = torch.where(ok, torch.where(last, t1, t + hc), t)
        grow = torch.where(e < 0.5, 0.9 * e.clamp(min=5.0 ** -8) ** -0.125,
                           torch.ones_like(e))
        h = torch.where(ok, hc * grow, h)
        h = torch.where(bad, hc * (0.9 * e.clamp(min=1e-300) ** (-1 / 6))
                        .clamp(min=0.2), h)
        live = live & ~(ok & last)
    return x, acc, rej


def observables(E, x):
    """Ground population, yield, excited population and norm."""
    W = torch.zeros(4, x.shape[0], dtype=torch.float64, device=x.device)
    W[0, 0], W[3] = 1.0, 1.0
    o = 0
    for e in E:
        n = len(e)
        if n > 2:
            W[1, o + 1:o + n - 1] = (e[1:n - 1] > THRESHOLD).double()
            W[2, o + 1:o + n - 1] = 1.0
        o += n
    return W @ (x.real ** 2 + x.imag ** 2)


def flat(x):
    return torch.view_as_real(x.t().contiguous()).reshape(x.shape[1], -1)


def exact(case, seed):
    c = case
    dev = "cuda"

    def member(blocks, P, k):
        E, D = operator(blocks, c["e_lo"], seed, k)
        x = states(E, P, seed, k + 1)
        return E, (lambda x, F: derivative(E, D, c["gauge"], x, F)), x

    E, f, x = member(c["blocks"], c["P"], 0)
    if c["kind"] in ("rhs", "rhs_device"):
        F = torch.tensor(rhs_fields(c, seed), device=dev)
        return flat(f(x, F)).reshape(-1)
    if c["kind"] == "fixed":
        F = torch.tensor(fields_fixed(c, seed), device=dev)
        h = torch.full((c["P"],), DT, dtype=torch.float64, device=dev)
        pop = []
        for k in range(c["steps"]):
            y, _, _ = attempt(f, x, h, h, lambda t: F[:, k])
            x = normalised(y)
            pop.append(x[0].real ** 2 + x[0].imag ** 2)
        return {"pop": torch.stack(pop, 1), "x": flat(x)}
    if c["kind"] == "adjoint":
        env = envelopes(c, seed).requires_grad_(True)
        field = Envelope(env, c["w"], c["span"], c["gauge"])
        t0 = torch.zeros(c["P"], dtype=torch.float64, device=dev)
        xT, acc, _ = controlled(f, x, t0, t0 + c["span"], c["tol"], field)
        n0 = len(E[0])
        J = (xT[:n0].real ** 2 + xT[:n0].imag ** 2).sum(0)
        (grad,) = torch.autograd.grad(J.sum(), env)
        return {"J": J.detach(), "grad": grad,
                "steps": acc.to(torch.int32)}
    out = []
    parts = [(E, f, x)]
    if c["kind"] == "multi":
        parts.append(member(c["blocks2"], c["P2"], 4))
    for E, f, x in parts:
        fs = [Field(c, p) for p in range(x.shape[1])]
        t0 = torch.tensor([start_time(c, g) for g in fs], dtype=torch.float64,
                          device=dev)

        def field(t, fs=fs):
            return torch.tensor([g(float(v)) for g, v in zip(fs, t.tolist())],
                                dtype=torch.float64, device=dev)
        with torch.no_grad():
            xT, acc, rej = controlled(f, x, t0, t0 + c["span"], c["tol"],
                                      field)
        out.append({"accepted": acc.long(), "rejected": rej.long(),
                    "obs": observables(E, xT), "x": flat(xT)})
    return out
