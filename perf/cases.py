"""The calls this library's speed is judged by, as a user's program makes them.

Every case is a plain dict; `prepare` makes what a program holds before the
call (the space, the workspaces, the captured step, the state on the GPU),
`run` makes the call through the package's public entry points, `exact` gives
the same results in 64 bits from plain torch and numpy.  Kinds:

product   hc = H C, one application of the many-body Hamiltonian
sil       one short-iterative-Lanczos step of the coefficients, in place
density   rho1, rho2 and rho1^-1 of a coefficient vector
step      one whole MCTDHB time step (orbitals, h and g, coefficients,
          density matrices), from a captured graph or enqueued call by call
many      one step of many unequal solves together (packed steps for the
          small ones, step graphs for the others)

Sizes: N bosons in M orbitals, NC = C(N + M - 1, M - 1) configurations.
Coefficients are complex normal, normalised; h is random Hermitian of scale 1
and g a random two-body tensor with the bosonic and Hermitian symmetries, or
both come from Hermite-Gauss orbitals on a grid.  The working folder is the
repository's root.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "1d-mctdhb_amd"))

import mctdhb_amd as amd  # noqa: E402

DEV = "cuda"


def listed():
    return [
        # a ground-state relaxation of the smallest usual kind: ten bosons in a
        # harmonic trap, the step replayed from its graph thousands of times
        {"name": "step_n10_m4", "kind": "step", "npar": 10, "norb": 4, "intervals": 256, "fft": True,
         "periodic": True, "imag": True, "graph": True, "lanczos": 5},
        # the same kind of job as a program without graphs makes it, by
        # Crank-Nicolson between walls on an odd grid
        {"name": "step_cn_n5_m5", "kind": "step", "npar": 5, "norb": 5, "intervals": 800, "fft": False,
         "periodic": False, "imag": True, "graph": False, "lanczos": 5},
        # real-time dynamics after a quench, six orbitals on a fine grid, the
        # coefficients in the mixed form (NC = 33,649)
        {"name": "step_real_n18_m6", "kind": "step", "npar": 18, "norb": 6, "intervals": 1024, "fft": True,
         "periodic": True, "imag": False, "graph": True, "lanczos": 5},
        # a parameter scan: unequal ground states advanced together
        {"name": "many_24", "kind": "many", "count": 24, "mix": 11},
        # the large spaces: long propagations spend their time in these steps
        {"name": "sil_mixed_n100_m5", "kind": "sil", "npar": 100, "norb": 5, "lanczos": 6, "mixed": True,
         "imag": False},
        {"name": "sil_fp64_n100_m5", "kind": "sil", "npar": 100, "norb": 5, "lanczos": 6, "mixed": False,
         "imag": False},
        {"name": "sil_mixed_n30_m7", "kind": "sil", "npar": 30, "norb": 7, "lanczos": 8, "mixed": True,
         "imag": False},
        {"name": "sil_mixed_n200_m4", "kind": "sil", "npar": 200, "norb": 4, "lanczos": 8, "mixed": True,
         "imag": False},
        # a middling space in imaginary time (NC = 23,751), all in FP64
        {"name": "sil_fp64_n25_m5", "kind": "sil", "npar": 25, "norb": 5, "lanczos": 5, "mixed": False, "imag": True},
        # one H C in FP64, as residuals and expectation values take it
        # (NC = 850,668)
        {"name": "product_fp64_n37_m6", "kind": "product", "npar": 37, "norb": 6, "mixed": False},
        # density matrices, in every step and for every observable
        {"name": "density_fp64_n100_m5", "kind": "density", "npar": 100, "norb": 5, "mixed": False},
        {"name": "density_mixed_n30_m7", "kind": "density", "npar": 30, "norb": 7, "mixed": True},
    ]


# Contraction work m P^2 C(N + M - 3, M - 1) of the largest listed steps.
MOST_FP64 = 6 * 225 * math.comb(102, 4)
MOST_MIXED = 8 * 784 * math.comb(34, 6)


def draw(rng):
    kind = rng.choice(["product", "sil", "sil", "density", "step", "step", "many"])
    if kind == "many":
        return {"kind": "many", "count": rng.randint(6, 24), "mix": rng.randint(1, 10 ** 6)}
    if kind == "step":
        fft = rng.random() < 0.6
        if fft and rng.random() < 0.7:
            intervals = rng.choice([128, 256, 512, 1024, 2048])
        else:
            intervals = int(round(math.exp(rng.uniform(math.log(100), math.log(700 if fft else 2000)))))
        while True:
            npar, norb = rng.randint(3, 64), rng.randint(2, 6)
            if _dim(npar, norb) <= 40000:
                break
        return {"kind": "step", "npar": npar, "norb": norb, "intervals": intervals, "fft": fft,
                "periodic": fft or rng.random() < 0.5, "imag": rng.random() < 0.6, "graph": rng.random() < 0.6,
                "lanczos": rng.randint(4, 8)}
    case = {"kind": kind, "mixed": rng.random() < 0.5}
    iters = rng.randint(4, 10) if kind == "sil" else 1
    most = MOST_MIXED if case["mixed"] else MOST_FP64
    while True:
        norb = rng.randint(2, 7)
        want = math.exp(rng.uniform(math.log(1e2), math.log(4.6e6)))
        npar = 2
        while npar < 4000 and _dim(npar + 1, norb) <= want:
            npar += 1
        if iters * _pairs(norb) ** 2 * _dim(npar - 2, norb) <= most:
            break
    case.update(npar=npar, norb=norb)
    if kind == "sil":
        case.update(lanczos=iters, imag=rng.random() < 0.5)
    return case


def _dim(npar, norb):
    return math.comb(npar + norb - 1, norb - 1)


def _pairs(norb):
    return norb * (norb + 1) // 2


# ------------------------------------------------------------------ inputs

def _normal(shape, seed, stream):
    """Complex normal numbers drawn on the GPU from the seed."""
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 16 + stream)
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.complex128)


def _coefficients(npar, norb, seed):
    c = _normal((_dim(npar, norb),), seed, 0)
    return c / torch.linalg.vector_norm(c)


def _matrices(npar, norb, seed):
    """Random Hermitian h and a two-body g with g[ksql] = g[skql] = g[kslq] =
    conj(g[lqsk]); g N stays at the scale of a trapped gas for large N."""
    a = _normal((norb, norb), seed, 1)
    h = 0.5 * (a + a.conj().T)
    g = min(0.1, 10.0 / npar) * _normal((norb,) * 4, seed, 2)
    g = g + g.permute(3, 2, 1, 0).conj()
    g = g + g.permute(1, 0, 2, 3)
    g = (g + g.permute(0, 1, 3, 2)) / 8
    # flat index k + s M + q M^2 + l M^3
    return h.contiguous().reshape(-1), g.permute(3, 2, 1, 0).contiguous().reshape(-1)


def _dt(npar):
    return 0.01 if npar <= 200 else 2.0 / npar


def _trap(case):
    """x, V(x), g, dt of a solve: a harmonic trap on [-8, 8], or the double
    well of a scan in the box where it reaches 200."""
    if "a" in case:
        a, b = case["a"], case["b"]
        half = min(10.0, math.sqrt(b * b + math.sqrt(200.0 / a)))
        x = np.linspace(-half, half, case["intervals"] + 1)
        return x, a * (x ** 2 - b ** 2) ** 2, case["g"], 0.005
    x = np.linspace(-8.0, 8.0, case["intervals"] + 1)
    return x, 0.5 * x ** 2, 1.0 if case["imag"] else 10.0 / case["npar"], 0.005 if case["imag"] else 0.002


def _orbitals(case, x, seed):
    """Hermite-Gauss functions with a little complex noise, as rows."""
    r = np.random.default_rng([seed, 3])
    out = np.zeros((case["norb"], x.size), complex)
    h0, h1 = np.zeros_like(x), np.exp(-x * x / 2) / math.pi ** 0.25
    for n in range(case["norb"]):
        out[n] = h1
        h0, h1 = h1, math.sqrt(2.0 / (n + 1)) * x * h1 - math.sqrt(n / (n + 1.0)) * h0
    out += 1e-3 * (r.standard_normal(out.shape) + 1j * r.standard_normal(out.shape))
    if case["periodic"]:
        out[:, -1] = out[:, 0]
    return out


def _members(case):
    """The solves of a `many` case: N in [4, 64], M in {2..6}, NC <= 2e5,
    256 to 1024 grid intervals, a double well and a contact interaction."""
    r = np.random.default_rng([case["mix"], 4])
    out = []
    while len(out) < case["count"]:
        npar, norb = int(r.integers(4, 65)), int(r.integers(2, 7))
        rest = {"intervals": int(r.choice([256, 512, 1024])), "a": float(r.uniform(0.5, 2.0)),
                "b": float(r.uniform(1.0, 3.0)), "g": float(10 ** r.uniform(-2.0, 1.0))}
        if _dim(npar, norb) <= 200_000:
            out.append({"npar": npar, "norb": norb, "fft": True, "periodic": True, "imag": True, "lanczos": 5, **rest})
    return out


# ----------------------------------------------------------------- prepare

class _Solve:
    """One solve: its handles and its state on the GPU."""

    def __init__(self, case, seed):
        npar, norb = case["npar"], case["norb"]
        x, pot, g, dt = _trap(case)
        # small spaces in FP64, larger ones in the mixed form
        prec = amd.FP64 if _dim(npar, norb) <= 8192 else amd.MIXED
        self.fft = case["fft"]
        self.space = amd.DeviceSpace(npar, norb, tables=False)
        self.sil = amd.DeviceSil(self.space, case["lanczos"], prec, amd.INDEX_FLY)
        self.orbital = amd.DeviceOrbital(norb, x.size, x[0], x[-1], dt, g, pot, imagtime=case["imag"],
                                         bounds=1001 if case["periodic"] else 1000)
        t = {"orb": torch.from_numpy(_orbitals(case, x, seed).reshape(-1)).to(DEV),
             "coef": _coefficients(npar, norb, seed)}
        for key, n in (("hob", norb ** 2), ("hint", norb ** 4), ("rho1", norb ** 2), ("rho2", norb ** 4),
                       ("rinv", norb ** 2)):
            t[key] = torch.zeros(n, dtype=torch.complex128, device=DEV)
        self.t = t
        self.orbital.orthonormalize(t["orb"])
        self.orbital.orbital_matrices(t["orb"], t["hob"], t["hint"])
        amd.density_sync(self.space, t["coef"], t["rho1"], t["rho2"], t["rinv"])

    def entry(self):
        t = self.t
        return (self.space, self.sil, self.orbital, t["orb"], t["coef"], t["hob"], t["hint"], t["rho1"], t["rho2"],
                t["rinv"])

    def graph(self):
        return amd.StepGraph(*self.entry(), use_fft=self.fft)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        s = _Solve(case, seed)
        return {"kind": kind, "solve": s, "graph": s.graph() if case["graph"] else None}
    if kind == "many":
        solves = [_Solve(m, seed * 64 + i) for i, m in enumerate(_members(case))]
        packed = [s for s in solves if amd.pack_eligible(s.space, s.sil, s.orbital)]
        alone = [s.graph() for s in solves if s not in packed]
        torch.cuda.synchronize()
        return {"kind": kind, "solves": solves, "pack": amd.Pack([s.entry() for s in packed]) if packed else None,
                "graphs": alone, "streams": [torch.cuda.Stream() for _ in range(8)],
                "pack_streams": [torch.cuda.Stream() for _ in range(8)]}
    npar, norb = case["npar"], case["norb"]
    prec = amd.MIXED if case["mixed"] else amd.FP64
    space = amd.DeviceSpace(npar, norb, tables=False)
    state = {"kind": kind, "space": space, "prec": prec, "c": _coefficients(npar, norb, seed)}
    if kind == "sil":
        state["h"], state["g"] = _matrices(npar, norb, seed)
        state["sil"] = amd.DeviceSil(space, case["lanczos"], prec, amd.INDEX_FLY)
        state["imag"] = case["imag"]
        state["dt"] = -1j * _dt(npar) if case["imag"] else _dt(npar)
        return state
    if case["mixed"]:
        state["c"] = state["c"].to(torch.complex64)
    if kind == "product":
        state["h"], state["g"] = _matrices(npar, norb, seed)
        state["out"] = torch.empty_like(state["c"])
    else:
        for key, n in (("rho1", norb ** 2), ("rho2", norb ** 4), ("rinv", norb ** 2)):
            state[key] = torch.zeros(n, dtype=torch.complex128, device=DEV)
    return state


# --------------------------------------------------------------------- run

def run(state):
    kind = state["kind"]
    if kind == "product":
        state["space"].apply_hamiltonian(state["c"], state["h"], state["g"], state["out"], state["prec"])
        return state["out"]
    if kind == "sil":
        state["sil"].step(state["c"], state["h"], state["g"], state["dt"], state["imag"])
        return state["c"]
    if kind == "density":
        amd.density_sync(state["space"], state["c"], state["rho1"], state["rho2"], state["rinv"], prec=state["prec"])
        return {"rho1": state["rho1"], "rho2": state["rho2"], "rinv": state["rinv"]}
    if kind == "step":
        s = state["solve"]
        if state["graph"] is not None:
            state["graph"].launch()
        else:
            amd.propagate_step(*s.entry(), use_fft=s.fft)
        return s.t
    if state["pack"] is not None:
        state["pack"].step(state["pack_streams"], 1)
    amd.launch_graphs(state["graphs"], state["streams"], 1)
    return [{"orb": s.t["orb"], "coef": s.t["coef"]} for s in state["solves"]]


# -------------------------------------------------------------------- work

def work(case):
    """Inputs read once, outputs written once; the operations are those of
    the two-body contraction over pairs (8 P^2 per configuration of N - 2
    particles, for H C and for rho2 alike), of the vector sums of the Lanczos
    recursion, and of the transforms, integrals and pointwise terms of the
    orbital step."""
    kind = case["kind"]
    if kind == "many":
        parts = [work({"kind": "step", **m}) for m in _members(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    npar, norb = case["npar"], case["norb"]
    dim, pairs = _dim(npar, norb), _pairs(norb)
    contract = 8 * pairs ** 2 * _dim(npar - 2, norb)
    small = 16 * (2 * norb ** 4 + 3 * norb ** 2)
    if kind == "product":
        return {"bytes": 2 * (8 if case["mixed"] else 16) * dim + small, "flops": contract}
    if kind == "density":
        return {"bytes": (8 if case["mixed"] else 16) * dim + small, "flops": contract}
    m = case["lanczos"]
    sil = m * contract + 8 * dim * (2 * m * (m - 1) + 2 * m)
    if kind == "sil":
        return {"bytes": 32 * dim + small, "flops": sil}
    n = case["intervals"]
    orbital = (norb * (20 * n * math.log2(n) if case["fft"] else 100 * n)  # two linear half steps
               + 2 * 8 * n * (pairs ** 2 + 2 * norb ** 2)                  # h and g, twice
               + 4 * 8 * n * norb ** 2 * pairs                             # four Runge-Kutta stages
               + 8 * n * norb ** 2)                                        # orthonormalisation
    return {"bytes": 32 * dim + 32 * norb * n + 2 * small, "flops": sil + contract + orbital}


def tolerance(case):
    """About four times what separates the results from the 64-bit ones below,
    the worst over the listed sizes and a hundred drawn ones."""
    kind = case["kind"]
    if kind == "product":
        return {"rel": 6e-7} if case["mixed"] else {"rel": 4e-15}
    if kind == "sil":
        return {"rel": 2e-6} if case["mixed"] else {"rel": 1e-14}
    if kind == "density":
        return {"rel": 5e-8} if case["mixed"] else {"rel": 4e-15}
    if kind == "step" and _dim(case["npar"], case["norb"]) <= 8192:
        return {"rel": 2e-14}
    return {"rel": 8e-7}  # the larger spaces' coefficients in the mixed form


# ------------------------------------------------------------------- exact

class _Fock:
    """Occupation rows of N particles in M orbitals in the library's order,
    and the ladder operators between neighbouring particle numbers.
    rank(n) = NC - 1 - sum_m C(P_m + m, m + 1), P_m = n_0 + ... + n_m."""

    def __init__(self, npar, norb):
        self.npar, self.norb, self.dim = npar, norb, _dim(npar, norb)
        self.w = [torch.tensor([math.comb(p + m, m + 1) for p in range(npar + 1)], device=DEV)
                  for m in range(norb - 1)]
        left = self.dim - 1 - torch.arange(self.dim, device=DEV)
        hi = torch.full((self.dim,), npar, device=DEV)
        self.n = [None] * norb
        for m in range(norb - 2, -1, -1):
            p = torch.minimum(torch.searchsorted(self.w[m], left, right=True) - 1, hi)
            left = left - self.w[m][p]
            self.n[m + 1] = hi - p
            hi = p
        self.n[0] = hi

    def rank(self, n):
        r = torch.full_like(n[0], self.dim - 1)
        p = torch.zeros_like(n[0])
        for m in range(self.norb - 1):
            p = (p + n[m]).clamp(max=self.npar)  # rows of another particle number stay in the table
            r = r - self.w[m][p]
        return r.clamp(min=0)


def _lower(up, low, c, k):
    """a_k c: from the space `up` (N) to `low` (N - 1)."""
    n = [x + (1 if j == k else 0) for j, x in enumerate(low.n)]
    return torch.sqrt(n[k].double()) * c[up.rank(n)]


def _raise(up, low, c, k):
    """a+_k c: from `low` (N - 1) to `up` (N); the factor is zero where n_k is."""
    n = [(x - 1).clamp(min=0) if j == k else x for j, x in enumerate(up.n)]
    return torch.sqrt(up.n[k].double()) * c[low.rank(n)]


class _Hamiltonian:
    """H C and the density matrices from a_q a_l C on N - 2 particles."""

    def __init__(self, npar, norb):
        self.up, self.mid = _Fock(npar, norb), _Fock(npar - 1, norb)
        self.low = _Fock(npar - 2, norb) if npar >= 2 else None
        self.norb = norb

    def pair_states(self, ones):
        return {(q, l): _lower(self.mid, self.low, ones[l], q)
                for q in range(self.norb) for l in range(q, self.norb)}

    def apply(self, c, h, g):
        m = self.norb
        h = h.reshape(m, m)
        g = g.reshape(m, m, m, m).permute(3, 2, 1, 0)  # g[k, s, q, l]
        ones = [_lower(self.up, self.mid, c, k) for k in range(m)]
        mid = [sum(h[k, l] * ones[l] for l in range(m)) for k in range(m)]
        if self.low is not None:
            phi = self.pair_states(ones)
            for k in range(m):
                for s in range(m):
                    psi = sum((g[k, s, q, l] if q == l else g[k, s, q, l] + g[k, s, l, q]) * phi[q, l]
                              for q, l in phi)
                    mid[k] = mid[k] + 0.5 * _raise(self.mid, self.low, psi, s)
        return sum(_raise(self.up, self.mid, mid[k], k) for k in range(m))

    def densities(self, c):
        m = self.norb
        ones = [_lower(self.up, self.mid, c, k) for k in range(m)]
        rho1 = torch.stack([torch.stack([torch.vdot(a, b) for b in ones]) for a in ones])
        rho2 = torch.zeros(m, m, m, m, dtype=torch.complex128, device=DEV)  # [l, q, s, k]
        if self.low is not None:
            phi = self.pair_states(ones)
            for (k, s), a in phi.items():
                for (q, l), b in phi.items():
                    v = torch.vdot(a, b)
                    for i, j in {(k, s), (s, k)}:
                        for u, w in {(q, l), (l, q)}:
                            rho2[w, u, j, i] = v
        return rho1.reshape(-1), rho2.reshape(-1)

    def sil(self, c, h, g, iters, dt, imag):
        """exp(-i H dt) c projected on the Krylov space of `iters` vectors."""
        v, alpha, beta = [c], [], []
        for it in range(iters):
            w = self.apply(v[it], h, g)
            alpha.append(float(torch.vdot(v[it], w).real))
            for _ in range(2):
                for u in v:
                    w = w - torch.vdot(u, w) * u
            if it == iters - 1 or v[0].numel() == len(v):
                break
            beta.append(float(torch.linalg.vector_norm(w)))
            v.append(w / beta[-1])
        d, z = np.linalg.eigh(np.diag(alpha) + np.diag(beta, 1) + np.diag(beta, -1))
        e = -1j * d * dt
        y = z @ (np.exp(e - (e.real.max() if imag else 0.0)) * z[0])
        out = sum(complex(y[k]) * v[k] for k in range(len(v)))
        return out / torch.linalg.vector_norm(out) if imag else out


def _simpson(n, dx):
    w = np.zeros(n)
    e = n - 1 if n % 2 else n - 4
    if e > 0:
        w[:e + 1] = 2 * dx / 3
        w[1:e:2] = 4 * dx / 3
        w[0] = w[e] = dx / 3
    if n % 2 == 0:
        w[e] += 3 * dx / 8
        w[n - 3:n - 1] += 9 * dx / 8
        w[n - 1] += 3 * dx / 8
    return w


def _orthonormalise(f, w):
    """Gram-Schmidt whose projection coefficient is taken anew at each point:
    at point p it has shrunk by prod_{q < p} (1 - w_q |F_j(q)|^2)."""
    for i in range(len(f)):
        for j in range(i):
            d = w * np.abs(f[j]) ** 2
            shrink = np.concatenate([[1.0], np.cumprod(1.0 - d)[:-1]])
            f[i] = f[i] - np.sum(w * f[j].conj() * f[i]) * shrink * f[j]
        f[i] = f[i] / math.sqrt(np.sum(w * np.abs(f[i]) ** 2))
    return f


def _orbital_matrices(f, w, dx, pot, g):
    """h[i, j] and g[a, b, c, d] = g int conj(f_a f_b) f_c f_d."""
    n = f.shape[1]
    core = f[:, :n - 1]  # the derivative takes the last point as the first
    df = (np.roll(core, 2, 1) - np.roll(core, -2, 1) + 8 * (np.roll(core, -1, 1) - np.roll(core, 1, 1))) / (12 * dx)
    df = np.concatenate([df, df[:, :1]], 1)
    h = (0.5 * df.conj() * w) @ df.T + (f.conj() * (w * pot)) @ f.T
    h = np.triu(h, 1) + np.triu(h, 1).conj().T + np.diag(np.diag(h).real)
    pair = (f[:, None] * f[None]).reshape(-1, n)
    return h, (g * (pair.conj() * w) @ pair.T).reshape((len(f),) * 4)


def _exact_step(case, seed):
    npar, norb = case["npar"], case["norb"]
    x, pot, g, dt = _trap(case)
    n, dx = x.size, x[1] - x[0]
    dx = (x[-1] - x[0]) / (n - 1)
    w = _simpson(n, dx)
    pdt = -1j * dt if case["imag"] else dt
    f = _orthonormalise(_orbitals(case, x, seed), w)
    many = _Hamiltonian(npar, norb)
    c = _coefficients(npar, norb, seed)

    def densities(c):
        r1, r2 = (t.cpu().numpy() for t in many.densities(c))
        r1 = r1.reshape(norb, norb)
        return r1, r2.reshape((norb,) * 4).transpose(3, 2, 1, 0), np.linalg.inv(r1)

    if case["fft"]:
        k = 2 * math.pi * np.fft.fftfreq(n - 1, dx)
        phase = np.exp(-0.5j * pdt * 0.5 * k * k)

        def linear(f):
            out = np.fft.ifft(phase * np.fft.fft(f[:, :n - 1], axis=1), axis=1)
            return np.concatenate([out, out[:, :1]], 1)
    else:
        m = n - 1 if case["periodic"] else n
        t = np.diag(np.full(m, -2.0)) + np.diag(np.ones(m - 1), 1) + np.diag(np.ones(m - 1), -1)
        if case["periodic"]:
            t[0, -1] = t[-1, 0] = 1.0
        t = -0.5 / dx ** 2 * t
        one = np.eye(m)
        cayley = np.linalg.solve(one + 0.25j * pdt * t, one - 0.25j * pdt * t)

        def linear(f):
            out = f[:, :m] @ cayley.T
            return np.concatenate([out, out[:, :1]], 1) if case["periodic"] else out

    _, r2, rinv = densities(c)
    f = linear(f)
    h, hint = _orbital_matrices(f, w, dx, pot, g)
    a = np.einsum("ka,asql->ksql", rinv, r2)
    proj = h.T + np.einsum("ksql,jslq->kj", a, hint)

    def rhs(y):
        cubic = np.einsum("ksx,sx->kx", np.einsum("ksql,qx,lx->ksx", a, y, y, optimize=True), y.conj())
        return -1j * (-1j if case["imag"] else 1.0) * (g * cubic + pot * y - proj @ y)

    k1 = rhs(f)
    k2 = rhs(f + 0.5 * dt * k1)
    k3 = rhs(f + 0.5 * dt * k2)
    k4 = rhs(f + dt * k3)
    f = linear(f + dt / 6 * (k1 + 2 * k2 + 2 * k3 + k4))
    if case["imag"]:
        f = _orthonormalise(f, w)
    if case["periodic"]:
        f[:, -1] = f[:, 0]
    h, hint = _orbital_matrices(f, w, dx, pot, g)
    flat = np.ascontiguousarray(hint.transpose(3, 2, 1, 0)).reshape(-1)
    c = many.sil(c, torch.from_numpy(h).to(DEV), torch.from_numpy(flat).to(DEV), case["lanczos"], pdt, case["imag"])
    r1, r2, rinv = densities(c)
    back = {"orb": f, "hob": h, "hint": flat, "rho1": r1, "rho2": np.ascontiguousarray(r2.transpose(3, 2, 1, 0)),
            "rinv": rinv}
    return {"coef": c, **{k: torch.from_numpy(np.ascontiguousarray(v).reshape(-1)) for k, v in back.items()}}


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return _exact_step(case, seed)
    if kind == "many":
        got = [_exact_step(m, seed * 64 + i) for i, m in enumerate(_members(case))]
        return [{"orb": s["orb"], "coef": s["coef"]} for s in got]
    npar, norb = case["npar"], case["norb"]
    many = _Hamiltonian(npar, norb)
    c = _coefficients(npar, norb, seed)
    if kind == "sil":
        h, g = _matrices(npar, norb, seed)
        dt = -1j * _dt(npar) if case["imag"] else _dt(npar)
        return many.sil(c, h, g, case["lanczos"], dt, case["imag"])
    if case["mixed"]:
        c = c.to(torch.complex64).to(torch.complex128)  # the call's input, in 64 bits
    if kind == "product":
        h, g = _matrices(npar, norb, seed)
        return many.apply(c, h, g)
    rho1, rho2 = many.densities(c)
    return {"rho1": rho1, "rho2": rho2, "rinv": torch.linalg.inv(rho1.reshape(norb, norb)).reshape(-1)}
