"""The work that users of the time-step library have it do, as measurable cases.

``listed()`` names the cases, ``draw(rng)`` gives further ones of the same
ranges, ``prepare``/``run`` take a case through the public entry points
(``opf.Context`` and ``opf.Server`` over the C ABI), ``work`` states the bytes
and operations that one pass cannot do without, and ``exact`` computes the
same results with dense linear algebra and library transforms in 64 bits,
without the library.

Kinds of work (``kind``):

dns        one state advanced by ``steps`` steps with the corrector iterated
           to convergence, then the state fetched: direct numerical
           simulation that writes a state every ``steps`` steps.  The state
           stays on the device between passes.
ensemble   the same for ``slots`` independent states in one context.
orbit      what a Newton-Krylov search does for each of its iterates: states
           loaded, integrated over their periods with one corrector a step
           (``steporbit``, new matrices for each period), shifted back and
           fetched; ``slots`` segments at once.
host       the loop of a Fortran host through the one-procedure entry points
           (transform, nonlinear, predictor, corrector), the corrector test
           on the host, then the state fetched.
serve      integration requests of mixed resolution, submitted at once to the
           request server and fetched as they finish.

Options of a state (``option``): none, adaptive (time step from the CFL limit,
matrices rebuilt where it changes), coriolis, shiftrefl / mirror / shiftrott
(symmetric subspaces), nonnewtonian (Carreau-Yasuda viscosity).
"""
import ctypes
import math
import os
import sys
import time

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "softx-d-17-00015_amd")

KL = 4
IMPLICIT = 0.51
DTERR_TOL = 1e-5
CORIOLIS = dict(Ek0=0.05, phi=0.6)
CARREAU = dict(rho=1.0, radius=1.0, mu_0=1.0, mu_inf=0.1, lam_CY=1e-3, n_CY=0.5, a_CY=2.0)


def _opf():
    if _PKG not in sys.path:
        sys.path.insert(0, _PKG)
    import opf
    return opf


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def _case(name, kind, N, K, M, steps, slots=1, Re=2400.0, alpha=1.25, dt=0.01, E0=1e-2, Mp=1, option="none"):
    return dict(name=name, kind=kind, N=N, K=K, M=M, Mp=Mp, slots=slots, steps=steps, Re=Re, alpha=alpha, dt=dt,
                E0=E0, option=option)


def listed():
    return [
        # a minimal flow unit at the smallest grid of the tests: launches and latency
        _case("dns_16_6_4", "dns", 16, 6, 4, 100, Re=1800.0),
        # the small grid of the benchmark's ensemble and of the drop-in host, one state
        _case("dns_32_24_12", "dns", 32, 24, 12, 200),
        # an odd radial resolution, lengths with no tuned launch shapes, three-fold symmetry, Coriolis is Mp = 1 only
        _case("dns_45_36_18_mp3", "dns", 45, 36, 18, 100, Re=2800.0, Mp=3),
        # the serving size with the time step chosen from the CFL limit
        _case("adaptive_48_48_24", "dns", 48, 48, 24, 100, Re=3000.0, option="adaptive"),
        # the benchmark's headline: transitional flow at (64, 64, 48)
        _case("dns_64_64_48", "dns", 64, 64, 48, 200, Re=5300.0, alpha=0.5, dt=0.005),
        # the benchmark's large size
        _case("dns_96_256_128", "dns", 96, 256, 128, 80, Re=5300.0, alpha=0.5, dt=0.0025),
        # the benchmark's ensemble: independent states in one context
        _case("ensemble_32_24_12", "ensemble", 32, 24, 12, 100, slots=64, Re=2400.0),
        # four shooting segments of a relative periodic orbit in the shift-reflect subspace
        _case("orbit_32_24_12", "orbit", 32, 24, 12, 100, slots=4, option="shiftrefl"),
        # the drop-in's host-driven loop
        _case("host_48_48_24", "host", 48, 48, 24, 25, Re=3000.0),
        # rotating pipe at an ordinary size
        _case("coriolis_64_32_24", "dns", 64, 32, 24, 100, Re=3000.0, option="coriolis"),
        # shear-thinning fluid
        _case("nonnewtonian_48_48_24", "dns", 48, 48, 24, 30, Re=3000.0, option="nonnewtonian"),
        # mixed requests at once
        _case("serve_mix", "serve", 64, 64, 48, 100, slots=16, alpha=1.25),
    ]


_KS = (6, 8, 9, 12, 16, 18, 24, 27, 32, 36, 48, 54, 64, 72, 81, 96, 128, 144, 192, 256)
_MS = (4, 6, 8, 9, 12, 16, 18, 24, 27, 32, 36, 48, 54, 64, 72, 96, 128)


def draw(rng):
    kind = rng.choice(["dns"] * 6 + ["ensemble"] * 3 + ["orbit"] * 2 + ["host"])
    while True:
        N = int(round(math.exp(rng.uniform(math.log(16), math.log(96.49)))))
        K, M = rng.choice(_KS), rng.choice(_MS)
        size = N * K * M
        if K >= M and size <= (96 * 256 * 128 if kind == "dns" else 64 * 64 * 48):
            break
    Mp = rng.choice([1, 1, 1, 2, 3, 4])
    slots = 1
    if kind == "ensemble":
        slots = rng.randint(4, 64)
        while slots * size > 64 * 64 * 48 * 6:
            slots = max(2, slots // 2)
    elif kind == "orbit":
        slots = rng.randint(1, 6)
    # passes of about 10 to 200 ms
    steps = int(max(10, min(150, 6e7 / (slots * size))))
    option = "none"
    if kind == "dns":
        options = ["none"] * 4 + ["adaptive", "shiftrefl", "mirror", "shiftrott"]
        if size <= 64 * 64 * 48:
            options += ["nonnewtonian"] + ["coriolis"] * (Mp == 1)
        option = rng.choice(options)
    elif kind == "orbit":
        option = rng.choice(["none", "shiftrefl"])
    if option == "nonnewtonian":
        steps = max(5, steps // 4)
    if kind == "host":
        steps = min(steps, 30)
    alpha = rng.choice([0.5, 1.0, 1.25, 1.7])
    dt = min(0.01, round(0.3 * 2 * math.pi / (alpha * 3 * K), 5))
    return dict(kind=kind, N=N, K=K, M=M, Mp=Mp, slots=slots, steps=steps, Re=float(rng.randint(1800, 5300)),
                alpha=alpha, dt=dt, E0=10 ** rng.uniform(-4, -2), option=option)


# ---------------------------------------------------------------------------
# inputs, made from the seed alone
# ---------------------------------------------------------------------------
def _harmonics(K, M):
    k = np.concatenate([np.arange(K)] + [np.arange(-(K - 1), K)] * (M - 1))
    m = np.concatenate([np.zeros(K, int)] + [np.full(2 * K - 1, j) for j in range(1, M)])
    return k, m


def _radial_points(N):
    """The default mesh: Chebyshev-like towards the wall, the first point half a spacing off the axis."""
    n_ = N + int(math.sqrt(N))
    r = 0.5 * (1.0 + np.cos(math.pi * (N - 1 - np.arange(N)) / n_))
    for _ in range(10):
        d = 1.5 * r[0] - 0.5 * r[1]
        r = r * (1.0 + d) - d
    return r


def _state(N, K, M, Mp, alpha, E0, rng):
    """A solenoidal no-slip perturbation, curl(psi z) + curl curl(phi z), with
    a Gaussian spectrum over the large scales: host planes (6, H, N)."""
    from numpy.polynomial import Polynomial as Poly
    r = _radial_points(N)
    k, m = _harmonics(K, M)
    u = np.zeros((3, N, k.size), complex)
    g = rng.standard_normal((4, k.size)) * np.exp(-(k * k + m * m) / 16.0)
    cpsi, cphi = g[0] + 1j * g[1], g[2] + 1j * g[3]
    cpsi[0], cphi[0] = cpsi[0].real, cphi[0].real
    for j in range(min(M, 25)):
        mm = j * Mp
        wall = Poly([1.0, 0.0, -1.0])
        psi, phi = wall ** 2, wall ** 3          # over r^mm
        x = Poly([0.0, 1.0])
        dpsi_r = mm * psi + x * psi.deriv()      # psi' = r^(mm-1) dpsi_r
        dphi_r = mm * phi + x * phi.deriv()
        lap = (2 * mm + 1) * phi.deriv() + x * phi.deriv().deriv()   # laplacian of phi = r^(mm-1) lap
        p = r ** (mm - 1.0)
        s = np.nonzero((m == j) & (np.abs(k) <= 24))[0]
        ak = alpha * k[s]
        a = lambda f: (p * f(r))[:, None]        # noqa: E731
        u[0][:, s] = 1j * mm * a(psi) * cpsi[s] + 1j * a(dphi_r) * (ak * cphi[s])
        u[1][:, s] = -a(dpsi_r) * cpsi[s] - mm * a(phi) * (ak * cphi[s])
        u[2][:, s] = -a(lap) * cphi[s]
    u[0][:, 0] = 0.0
    u[1:, :, 0] = u[1:, :, 0].real
    dr = np.gradient(r) * r
    energy = 4 * math.pi ** 2 / alpha * np.einsum("cnh,n->", np.abs(u) ** 2, dr)
    u *= math.sqrt(E0 / energy)
    return np.ascontiguousarray(np.stack([u.real, u.imag], 1).reshape(6, N, -1).transpose(0, 2, 1))


def _members(case, seed):
    """(planes, Re, dt, T, shifts) of every state of a case."""
    rng = np.random.default_rng([int(seed), 71])
    got = []
    for i in range(case["slots"]):
        f = 1.0 if i == 0 else rng.uniform(0.85, 1.15)
        dt = case["dt"]
        u = _state(case["N"], case["K"], case["M"], case["Mp"], case["alpha"], case["E0"] * f * f, rng)
        got.append(dict(u=u, Re=case["Re"] * f, dt=dt, T=dt * case["steps"] * rng.uniform(0.9, 1.0),
                        sth=rng.uniform(-0.1, 0.1), sz=rng.uniform(-0.5, 0.5)))
    if case["option"] in ("shiftrefl", "mirror", "shiftrott"):
        for g in got:
            _impose(g["u"], case, case["option"])
    return got


def _image(K, M, k, m):
    at = {(int(a), int(b)): i for i, (a, b) in enumerate(zip(k, m))}
    return np.array([i if m[i] == 0 else at[(-int(k[i]), int(m[i]))] for i in range(k.size)])


def _impose(u, case, option):
    """The symmetry on host planes, so that runs start inside their subspace."""
    k, m = _harmonics(case["K"], case["M"])
    if option == "shiftrott":
        u[:, (k + m) % 2 != 0] = 0.0
        return
    img = _image(case["K"], case["M"], k, m)
    a = np.where((k % 2 != 0) & (option == "shiftrefl"), -1.0, 1.0)
    b = np.where(m == 0, 1.0, -1.0)
    for c, s in ((0, 1.0), (1, -1.0), (2, 1.0)):
        u[2 * c] = 0.5 * (u[2 * c] + u[2 * c][img] * (s * a)[:, None])
        u[2 * c + 1] = 0.5 * (u[2 * c + 1] + u[2 * c + 1][img] * (s * a * b)[:, None])


# ---------------------------------------------------------------------------
# what a user's program holds, and one pass
# ---------------------------------------------------------------------------
def _ptrs(planes):
    return [p.ctypes.data_as(ctypes.POINTER(ctypes.c_double)) for p in planes]


def _ok(ctx, rc):
    if rc:
        raise RuntimeError(ctx.lib.opf_last_error().decode())


def _put(ctx, slot, planes):
    """A host in the coll layout (the Fortran arrays) loads its state."""
    _ok(ctx, ctx.lib.opf_put_state(ctx.h, slot, *_ptrs(planes), 0.0))


def _get(ctx, slot, planes):
    t = ctypes.c_double()
    _ok(ctx, ctx.lib.opf_get_state(ctx.h, slot, *_ptrs(planes), ctypes.byref(t)))
    return planes


# the request mix of the benchmark's serving part: class, steps of each request
_CLASSES = ((32, 24, 12), (48, 48, 24), (64, 64, 48))


def _requests(case, seed):
    rng = np.random.default_rng([int(seed), 72])
    got = []
    for i in range(case["slots"]):
        c = (0, 1, 0, 2, 0, 1, 0, 1, 0, 2)[i % 10]
        n, k, m = _CLASSES[c]
        alpha = float(rng.choice([0.5, 1.25]))
        got.append(dict(cls=c, Re=float(rng.uniform(2000, 5300)), alpha=alpha,
                        steps=int(case["steps"] * (1 + i % 4)) // (1 + c),
                        u=_state(n, k, m, 1, alpha, case["E0"] * 0.1, rng)))
    return got


def prepare(case, seed):
    opf = _opf()
    if case["kind"] == "serve":
        reqs = _requests(case, seed)
        fields = [[np.ascontiguousarray((q["u"][2 * c] + 1j * q["u"][2 * c + 1]).T) for c in range(3)] for q in reqs]
        srv = opf.Server(list(_CLASSES), [8, 4, 2], 16 << 30, depth=3)
        return dict(case=case, srv=srv, reqs=reqs, fields=fields)
    ctx = opf.Context(case["N"], case["K"], case["M"], case["Mp"], capacity=case["slots"])
    members = _members(case, seed)
    for i, g in enumerate(members):
        option = case["option"]
        if option in ("mirror", "shiftrefl", "shiftrott"):
            ctx.symmetry(i, **{option: True})
        elif option == "adaptive":
            ctx.adaptive(i, True)
        elif option == "coriolis":
            ctx.coriolis(i, **CORIOLIS)
        elif option == "nonnewtonian":
            ctx.nonnewtonian(i, **CARREAU)
        ctx.setup(i, g["Re"], case["alpha"], g["dt"], implicit=IMPLICIT)
        _put(ctx, i, g["u"])
    out = [np.zeros_like(g["u"]) for g in members]
    return dict(case=case, ctx=ctx, members=members, out=out)


def run(state):
    case = state["case"]
    return {"dns": _run_loop, "ensemble": _run_loop, "orbit": _run_orbit, "host": _run_host,
            "serve": _run_serve}[case["kind"]](state, case)


def _run_loop(state, case):
    ctx = state["ctx"]
    ctx.run(case["steps"])
    return [_get(ctx, i, o) for i, o in enumerate(state["out"])]


def _run_orbit(state, case):
    ctx, members = state["ctx"], state["members"]
    n = len(members)
    for i, g in enumerate(members):
        _put(ctx, i, g["u"])
    ctx.steporbit(range(n), case["steps"], [g["T"] for g in members], [g["sth"] for g in members],
                  [g["sz"] for g in members])
    return [_get(ctx, i, o) for i, o in enumerate(state["out"])]


def _run_host(state, case):
    ctx = state["ctx"]
    for _ in range(case["steps"]):
        ctx.imposesym(0)
        ctx.transform(0)
        ctx.nonlinear(0)
        ctx.predictor(0)
        for _ in range(10):
            ctx.transform(0)
            ctx.nonlinear(0)
            if ctx.corrector(0) <= DTERR_TOL:
                break
    return [_get(ctx, 0, state["out"][0])]


def _run_serve(state, case):
    srv = state["srv"]
    ids = [srv.submit(q["cls"], q["Re"], q["alpha"], 0.01, q["steps"], f)
           for q, f in zip(state["reqs"], state["fields"])]
    out = []
    for rid, q in zip(ids, state["reqs"]):
        while True:
            p = srv.poll(rid)
            if p["done"]:
                break
            time.sleep(2e-4)
        if p["status"]:
            raise RuntimeError("request failed")
        out.append(np.stack(srv.result(rid, q["cls"])[:3]))
    return out


def _per_step(N, K, M, corr):
    """Bytes and flops of a step that iterates `corr` correctors: per
    evaluation u and curl u in, N out (9 C); the predictor reads N and u and
    writes u and curl u (12 C), a corrector also reads the predictor's N and
    the last iterate (18 C); both read the factors of the four systems of a
    (|k|, m) pair and the influence vectors.  Flops: the transforms' 5 L log2 L
    and the band solves."""
    H = (2 * K - 1) * M - (K - 1)
    P, Z, T = K * M, 3 * K, 3 * M
    C = 16.0 * N * H
    F = 4 * P * N * 13 * 8 + H * (6 * 8 * N + 128)
    evals = 1 + corr
    byts = (9 + 12) * C + corr * (9 + 18) * C + evals * F
    line = N * (9 * M * 5 * Z * math.log2(Z) + 9 * Z * 2.5 * T * math.log2(T))
    flops = evals * (line + H * N * (4 * 2 * 2 * 13 + 3 * 9 * 4 * 4))
    return byts, flops


def work(case):
    if case["kind"] == "serve":
        parts = [(_CLASSES[q["cls"]], q["steps"]) for q in
                 [dict(cls=(0, 1, 0, 2, 0, 1, 0, 1, 0, 2)[i % 10],
                       steps=int(case["steps"] * (1 + i % 4)) // (1 + (0, 1, 0, 2, 0, 1, 0, 1, 0, 2)[i % 10]))
                  for i in range(case["slots"])]]
    else:
        parts = [((case["N"], case["K"], case["M"]), case["steps"])] * case["slots"]
    b = f = 0.0
    for (N, K, M), steps in parts:
        sb, sf = _per_step(N, K, M, 1)
        if case["option"] == "nonnewtonian":   # 9 gradients, nu, 3 of grad nu, 3 of curl curl, 3 forces
            H = (2 * K - 1) * M - (K - 1)
            sb += 2 * 2 * 16.0 * N * H * 3
            sf += 2 * N * 19 * (M * 5 * 3 * K * math.log2(3 * K) + 3 * K * 2.5 * 3 * M * math.log2(3 * M))
        b += steps * sb
        f += steps * sf
        b += 6 * 8.0 * N * ((2 * K - 1) * M - (K - 1)) * (2 if case["kind"] in ("orbit", "serve") else 1)
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------
# the same results in 64 bits from dense matrices and library transforms
# ---------------------------------------------------------------------------
def _weights(i, x, x0):
    """Weights of the i-th derivative at x0 of the polynomial through x."""
    lo, hi = min(x0, x.min()), max(x0, x.max())
    t, t0 = (2 * x - lo - hi) / (hi - lo), (2 * x0 - lo - hi) / (hi - lo)
    V = np.polynomial.chebyshev.chebvander(t, x.size - 1)
    d = np.array([np.polynomial.chebyshev.Chebyshev.basis(j).deriv(i)(t0) if i else
                  np.polynomial.chebyshev.Chebyshev.basis(j)(t0) for j in range(x.size)])
    return np.linalg.solve(V.T, d) * (2.0 / (hi - lo)) ** i


class _Exact:
    """Pressure-projection predictor-corrector for one state: dense radial
    operators, explicit inverses with one refinement, torch FFTs."""

    def __init__(self, case, N, K, M, Mp, Re, alpha, dt, option="none"):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.N, self.K, self.M, self.Mp, self.Re, self.alpha, self.dt = N, K, M, Mp, Re, alpha, dt
        self.option = option
        k, m = _harmonics(K, M)
        self.kn, self.mn = k, m
        t = lambda a: torch.as_tensor(a, dtype=torch.float64, device=self.dev)   # noqa: E731
        r = _radial_points(N)
        D1, D2 = np.zeros((N, N)), np.zeros((N, N))
        r0 = np.concatenate([[0.0], r])
        quad = np.zeros(N)
        for n in range(N):
            a, b = max(0, n - KL), min(n + KL, N - 1) + 1
            D1[n, a:b], D2[n, a:b] = _weights(1, r[a:b], r[n]), _weights(2, r[a:b], r[n])
            c = e = 1.0
            for i in range(b - a):
                c *= (r0[min(n + 2, N)] - r[n]) / (i + 1)
                e *= (r0[n] - r[n]) / (i + 1)
                quad[a:b] += 0.5 * (c - e) * _weights(i, r[a:b], r[n]) * r[n]
        self.axis = [_weights(i, r[:KL + 1], 0.0) for i in (0, 1)]
        self.wall = [_weights(i, r[N - KL - 1:], 1.0 * r[-1]) for i in (0, 1)]
        self.lapn = D2 + D1 / r[:, None]
        self.r, self.rn = t(r), r
        self.D1, self.lap, self.quad = t(D1), t(self.lapn), t(quad)
        self.D1c = self.D1.to(torch.complex128)
        self.wall1 = t(self.wall[1])
        self.U = 1.0 - self.r ** 2
        self.k, self.m = t(k), t(m * Mp)
        self.ak = alpha * self.k
        self.mr = self.m[None, :] / self.r[:, None]
        self.t, self.step, self.corr_dt, self.ntc = 0.0, 0, 0.0, 0
        self.img = None
        if option in ("mirror", "shiftrefl"):
            self.img = torch.as_tensor(_image(K, M, k, m), device=self.dev)
        pos = np.concatenate([(k % (3 * K)) * M + m])
        self.pos = torch.as_tensor(pos, device=self.dev)
        self.matrices()

    def diag(self, pm):
        r2 = 1.0 / self.r ** 2
        d = -(r2[:, None] * self.m ** 2) - self.ak ** 2
        if pm:
            d = d - r2[:, None] * (1.0 + 2.0 * pm * self.m)
        return d          # (N, H)

    def system(self, pm, bc, c1, c2):
        """Dense matrices (H, N, N) with the axis and wall rows."""
        N, H = self.N, self.k.numel()
        A = (c2 * self.lap).repeat(H, 1, 1)
        i = torch.arange(N, device=self.dev)
        A[:, i, i] += (c2 * self.diag(pm) + c1).T
        odd = torch.as_tensor((self.mn * self.Mp + abs(pm)) % 2 == 1, device=self.dev)
        ax = [torch.as_tensor(w, device=self.dev) for w in self.axis]
        A[:, 0] = 0.0
        A[:, 0, :KL + 1] = torch.where(odd[:, None], ax[0][None], ax[1][None])
        A[:, N - 1] = 0.0
        A[:, N - 1, N - KL - 1:] = torch.as_tensor(self.wall[bc], device=self.dev)
        if bc == 1:
            A[0] = torch.eye(N, device=self.dev, dtype=torch.float64)
        s = 1.0 / A.abs().amax(dim=2, keepdim=True)
        B = A * s
        return B, torch.linalg.inv(B), s

    def solve(self, S, b, neumann=False):
        A, Ai, s = S
        x = torch.view_as_real(b.T.contiguous()).contiguous() * s
        y = torch.bmm(Ai, x)
        y = y + torch.bmm(Ai, x - torch.bmm(A, y))
        out = torch.view_as_complex(y.contiguous()).T.contiguous()
        if neumann:
            out[:, 0] = 0.0
        return out

    def matrices(self):
        d2 = -IMPLICIT / self.Re
        c1 = 1.0 / self.dt
        if not hasattr(self, "LN"):
            self.LN = self.system(0, 1, 0.0, 1.0)
        self.LD = [self.system(pm, 0, c1, d2) for pm in (1, -1, 0)]
        ui = torch.ones((self.N, self.k.numel()), dtype=torch.complex128, device=self.dev)
        ui[0] = ui[-1] = 0.0
        self.Ui = self.solve(self.LD[2], ui)[:, 0].real.clone()
        self.flux = 2.0 * (self.Ui @ self.quad)
        N = self.N
        z = lambda: torch.zeros((N, self.k.numel()), dtype=torch.complex128, device=self.dev)   # noqa: E731
        cols, vec = [], []
        for j in range(4):
            v = [z(), z(), z()]
            if j < 3:
                v[j][-1] = 1.0 if j < 2 else 1j
                v[j] = self.solve(self.LD[j], v[j])
            else:
                p = z()
                p[-1] = -1.0
                v = list(self.pm(*self.grad(self.solve(self.LN, p, True))))
            vec.append(v)
            cols.append(self.residual(*v).real)
        A = torch.stack(cols, 2).permute(1, 0, 2).contiguous()   # (H, 4, 4)
        A[0] = torch.eye(4, dtype=torch.float64, device=self.dev)
        self.vec, self.inf = vec, torch.linalg.inv(A)

    def pm(self, r, t, *z):
        return (r + 1j * t, r - 1j * t, *z)

    def rt(self, p, m):
        return 0.5 * (p + m), -0.5j * (p - m)

    def grad(self, p):
        return self.D1c @ p, 1j * self.mr * p, 1j * self.ak * p

    def div(self, r, t, z):
        return r / self.r[:, None] + self.D1c @ r + 1j * self.mr * t + 1j * self.ak * z

    def curl(self, r, t, z):
        return (1j * self.mr * z - 1j * self.ak * t, 1j * self.ak * r - self.D1c @ z,
                t / self.r[:, None] + self.D1c @ t - 1j * self.mr * r)

    def residual(self, p, m, z):
        """No-slip and divergence at the wall, (4, H); u_z times -i, so that the influence matrix is real."""
        r, t = self.rt(p, m)
        w = self.wall1.to(torch.complex128)
        dv = r[-1] / self.r[-1] + w @ r[self.N - KL - 1:] + 1j * self.mr[-1] * t[-1] + 1j * self.ak * z[-1]
        return torch.stack([p[-1], m[-1], -1j * z[-1], dv])

    def phys(self, a):
        N, K, M = self.N, self.K, self.M
        X = torch.zeros((N, 3 * K * M), dtype=torch.complex128, device=self.dev)
        X[:, self.pos] = a
        X = X.view(N, 3 * K, M)
        X[:, 2 * K + 1:, 0] = X[:, 1:K, 0].flip(1).conj()
        Y = torch.fft.ifft(X, dim=1, norm="forward")
        S = torch.zeros((N, 3 * K, 3 * M // 2 + 1), dtype=torch.complex128, device=self.dev)
        S[:, :, :M] = Y
        S[:, :, 0].imag = 0.0
        return torch.fft.irfft(S, n=3 * M, dim=2, norm="forward")

    def spec(self, p):
        Y = torch.fft.rfft(p, dim=2, norm="forward")[:, :, :self.M]
        return torch.fft.fft(Y, dim=1, norm="forward").reshape(self.N, -1)[:, self.pos].contiguous()

    def impose(self):
        u = self.u
        if self.option == "shiftrott":
            odd = torch.as_tensor((self.kn + self.mn) % 2 != 0, device=self.dev)
            u = [torch.where(odd, 0.0, f) for f in u]
        elif self.img is not None:
            a = torch.where((self.k % 2 != 0) & (self.option == "shiftrefl"), -1.0, 1.0).to(torch.float64)
            b = torch.as_tensor(np.where(self.mn == 0, 1.0, -1.0), device=self.dev)
            im = lambda f, s: torch.complex(f.real * (s * a), f.imag * (s * a * b))   # noqa: E731
            u = [0.5 * (f + im(f[:, self.img], s)) for f, s in zip(u, (1.0, -1.0, 1.0))]
        self.u = [f.clone() for f in u]
        self.u[0][:, 0] = 0.0
        for f in self.u[1:]:
            f[:, 0] = f[:, 0].real.to(torch.complex128)

    def evaluate(self):
        u = self.u
        v = [self.phys(f) for f in u]
        w = [self.phys(f) for f in self.curl(*u)]
        self.v = v
        n = [v[1] * w[2] - v[2] * w[1], v[2] * w[0] - v[0] * w[2], v[0] * w[1] - v[1] * w[0]]
        if self.option == "coriolis":
            th = 2 * math.pi / (3 * self.M) * torch.arange(3 * self.M, device=self.dev, dtype=torch.float64)
            d = -1.0 / (4.0 * self.Re * CORIOLIS["Ek0"])
            s, c = math.sin(CORIOLIS["phi"]), math.cos(CORIOLIS["phi"])
            o = (s * torch.cos(th), -s * torch.sin(th), c)
            z = v[2] + self.U[:, None, None]
            n = [n[0] + d * (o[1] * z - o[2] * v[1]), n[1] + d * (o[2] * v[0] - o[0] * z),
                 n[2] + d * (o[0] * v[1] - o[1] * v[0])]
        n = [self.spec(f) for f in n]
        adv = -1j * self.ak * self.U[:, None]
        n = [f + adv * g for f, g in zip(n, u)]
        n[2] = n[2] + 2.0 * self.r[:, None] * u[0]
        self.Pr0 = (u[2][self.N - KL - 1:, 0].real @ self.wall1) / -2.0
        n[2][:, 0] += 4.0 * self.Pr0 / self.Re
        if self.option == "nonnewtonian":
            n = [f + g for f, g in zip(n, self.shear_thinning())]
        self.n = n

    def shear_thinning(self):
        r, t, z = self.u[0], self.u[1], self.u[2].clone()
        z[:, 0] += self.U
        ri = 1.0 / self.r[:, None]
        im, ik = 1j * self.m[None, :], 1j * self.ak[None, :]
        g = [[self.D1c @ f for f in (r, t, z)],
             [ri * (im * r - t), ri * (im * t + r), ri * (im * z)],
             [ik * f for f in (r, t, z)]]
        A = [[self.phys(f) for f in row] for row in g]
        S = [[0.5 * (A[i][j] + A[j][i]) for j in range(3)] for i in range(3)]
        sr = torch.sqrt(2.0 * sum(S[i][j] ** 2 for i in range(3) for j in range(3)))
        q = CARREAU
        lam = self.Re * q["lam_CY"] * q["mu_0"] / (q["rho"] * q["radius"] ** 2)
        d = q["mu_inf"] / q["mu_0"]
        nu = d + (1.0 - d) * (1.0 + (lam * sr) ** q["a_CY"]) ** (-q["n_CY"] / q["a_CY"])
        gn = [self.phys(f) for f in self.grad(self.spec(nu))]
        cc = [self.phys(f) for f in self.curl(*self.curl(r, t, z))]
        return [self.spec(((1.0 - nu) * cc[i] + 2.0 * sum(gn[j] * S[j][i] for j in range(3))) / self.Re)
                for i in range(3)]

    def advance(self, base, n):
        """One solve of the pressure-projection scheme from u_ = base."""
        c1, c2 = 1.0 / self.dt, (1.0 - IMPLICIT) / self.Re
        lap = self.lap.to(torch.complex128)
        q = [f + c2 * (lap @ b + self.diag(pm) * b) + c1 * b
             for f, b, pm in zip(self.pm(*n), self.pm(*base), (1, -1, 0))]
        d = self.div(*self.rt(q[0], q[1]), q[2])
        d[0] = d[-1] = 0.0
        g = self.pm(*self.grad(self.solve(self.LN, d, True)))
        q = [a - b for a, b in zip(q, g)]
        for f in q:
            f[0] = f[-1] = 0.0
        q = [self.solve(L, f) for L, f in zip(self.LD, q)]
        res = self.residual(*q)
        a = -torch.einsum("hij,jh->ih", self.inf.to(torch.complex128), res)
        a[:, 0] = 0.0
        for c in range(3):
            q[c] = q[c] + sum(a[j] * self.vec[j][c] for j in range(4))
        r, t = self.rt(q[0], q[1])
        z = q[2]
        z[:, 0] += -(2.0 * (z[:, 0].real @ self.quad)) / self.flux * self.Ui
        r[:, 0] = 0.0
        t[:, 0] = t[:, 0].real.to(torch.complex128)
        z[:, 0] = z[:, 0].real.to(torch.complex128)
        self.u = [r, t, z]

    def cfl(self):
        d = np.gradient(self.rn)
        gap = np.diff(self.rn)
        d[0], d[-1] = gap[0], gap[-1]
        d[1:-1] = np.minimum(gap[:-1], gap[1:])
        dr = torch.as_tensor(d, device=self.dev)
        mx = [f.abs().amax(dim=(1, 2)) for f in (self.v[0], self.v[1], self.v[2] + self.U[:, None, None])]
        lim = [dr / mx[0], 2 * math.pi / (3 * self.M * self.Mp) / mx[1],
               2 * math.pi / (self.alpha * 3 * self.K) / mx[2]]
        return min(float(x.min()) for x in lim)

    def new_dt(self):
        cfl = self.cfl()
        dt = self.dt * 1.11
        if self.step == 0 and self.corr_dt == 0.0:
            dt = min(dt, cfl * 0.1)
        dt = min(dt, cfl * 0.5)
        if self.corr_dt > 0.0:
            dt = min(dt, self.corr_dt * 0.95)
        self.ntc -= 1
        if dt < self.dt * 0.95 or (dt > self.dt * 1.10 and self.ntc < 0):
            if dt >= self.dt:
                self.ntc = 99
            self.dt = dt
            self.matrices()

    def integrate(self, planes, steps, corr=0, simple=False):
        """`steps` steps from host planes; corr: correctors per step (0: to
        convergence); simple: the host loop's test alone."""
        u = torch.as_tensor(planes, device=self.dev).transpose(1, 2).reshape(3, 2, self.N, -1)
        self.u = [torch.complex(f[0].contiguous(), f[1].contiguous()) for f in u]
        if self.option == "nonnewtonian":
            corr = 1
        for _ in range(steps):
            self.impose()
            self.evaluate()
            if self.option == "adaptive":
                self.new_dt()
            base, first = self.u, self.n
            self.advance(base, first)
            it, last = 1, 1e99
            while True:
                before = self.u
                self.evaluate()
                n = [IMPLICIT * a + (1.0 - IMPLICIT) * b for a, b in zip(self.n, first)]
                self.advance(base, n)
                err = float(max((a - b).abs().max() for a, b in zip(self.u, before)))
                if it == 1:
                    self.corr_dt = self.dt * math.sqrt(DTERR_TOL / err) if err > 0 else 0.0
                if (corr and it >= corr) or (simple and (err <= DTERR_TOL or it >= 10)):
                    break
                if not corr and not simple:
                    if err > last:
                        self.corr_dt = self.dt / 5.0
                        break
                    if err <= DTERR_TOL:
                        break
                it, last = it + 1, err
            self.step += 1

    def shift(self, dth, dz):
        ph = torch.exp(-1j * (self.ak * dz + self.m * dth).to(torch.complex128))
        self.u = [f * ph for f in self.u]

    def planes(self):
        f = torch.stack([p for f in self.u for p in (f.real, f.imag)])
        return f.transpose(1, 2).contiguous().cpu().numpy()


def _cost(N, K, M, steps):
    """Seconds of an exact integration, roughly."""
    H = (2 * K - 1) * M
    return 2 * steps * (4e-3 + N * 9 * K * M * 6e-9 + H * N * N * 1e-10) + H * N * N * 5e-8


def exact(case, seed):
    if not torch.cuda.is_available() and case["N"] * case["K"] * case["M"] > 20000:
        return None
    if case["kind"] == "serve":
        out, spent = [], 0.0
        for q in _requests(case, seed):
            n, k, m = _CLASSES[q["cls"]]
            spent += _cost(n, k, m, q["steps"])
            if spent > 8.0:
                out.append(None)
                continue
            e = _Exact(case, n, k, m, 1, q["Re"], q["alpha"], 0.01)
            e.integrate(q["u"], q["steps"], corr=1)
            out.append(torch.stack(e.u).cpu().numpy())
        return out if any(x is not None for x in out) else None
    N, K, M = case["N"], case["K"], case["M"]
    H = (2 * K - 1) * M
    one = _cost(N, K, M, case["steps"]) * (3.0 if case["option"] == "nonnewtonian" else 1.0)
    if one > 12.0 or H * N * N * 8.0 > 4e9:
        return None          # over the time or the memory of dense matrices
    out = []
    for i, g in enumerate(_members(case, seed)):
        if i * one > 8.0 or i >= 3:
            out.append(None)   # a few of an ensemble's states stand for the rest
            continue
        e = _Exact(case, N, K, M, case["Mp"], g["Re"], case["alpha"],
                   g["T"] / case["steps"] if case["kind"] == "orbit" else g["dt"], case["option"])
        e.integrate(g["u"], case["steps"], corr=1 if case["kind"] == "orbit" else 0, simple=case["kind"] == "host")
        if case["kind"] == "orbit":
            e.impose()
            e.shift(-g["sth"], -g["sz"])
        out.append(e.planes())
    return out
