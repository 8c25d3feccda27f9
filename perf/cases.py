"""The work that users of the propagator have it do, at the sizes they do it.

Each case is one call (or one step's calls) of the public Python interface `gade.Propagator` on couplings written
by `couplings.generate`:

  apply         f(t) of a step, then y = (S + H(t)) x: the operator a program's own solver calls
  precondition  x = P^{-1} b, the block preconditioner
  run           Crank-Nicolson steps of one state in the middle of its pulse
  scan          the same for a batch of pulses that share the couplings
  assembled     the reference's formulation: assemble H(t) as CSR, then y = (S + H(t)) x
  populations   bound / ionised populations of a state by eigen-projection
  guess_grad    loss and gradient of the learned initial guess's network over a batch of training samples

A program loads a set of couplings once and then propagates many states and pulses with it, so the model (and what
it sets up once: preconditioner, eigenpairs, network) is kept per configuration; the states, pulses and training
samples are made from the seed.
"""
import atexit
import math
import os
import shutil
import struct
import tempfile

import numpy as np
import torch

from dirac_hydrogen_code_amd import gade
from dirac_hydrogen_code_amd.couplings import generate

SOL = 137.035999084  # speed of light, atomic units
OMEGA = 50.0         # carrier of the coupling files' Bessel kernels
RBOX = 30.0

DIPOLE = dict(nsplines=50, nkappa=4, nmu=0, nl=1, cycles=1, per_cycle=200)
PRODUCTION = dict(nsplines=250, nkappa=16, nmu=8, nl=8, cycles=15, per_cycle=533)
MIDDLE = dict(nsplines=100, nkappa=8, nmu=4, nl=4, cycles=4, per_cycle=400)
ODD = dict(nsplines=33, nkappa=5, nmu=0, nl=3, cycles=2, per_cycle=300)
TOL = 1e-12


def listed():
    return [
        # the smallest call: one operator product at the dipole size, where launches and latency are all there is
        dict(name="apply_dipole", call="apply", **DIPOLE),
        # the operator product of the production runs (204,000 unknowns)
        dict(name="apply_production", call="apply", **PRODUCTION),
        # the preconditioner solve of the production runs
        dict(name="precondition_production", call="precondition", **PRODUCTION),
        # a short pulse in the dipole approximation, one state: a window of steps between two outputs
        dict(name="run_dipole", call="run", steps=100, precision=0, guess=0, **DIPOLE),
        # the production run at the middle of its pulse, all in FP64
        dict(name="run_production", call="run", steps=16, precision=0, guess=0, **PRODUCTION),
        # the same with FP32 inner solves under FP64 defect correction
        dict(name="run_production_mixed", call="run", steps=8, precision=1, guess=0, **PRODUCTION),
        # a scan over pulses at the dipole size
        dict(name="scan_dipole_64", call="scan", batch=64, steps=40, precision=0, guess=0, **DIPOLE),
        # a small scan with odd sizes, started from the extrapolated guess
        dict(name="scan_odd_5", call="scan", batch=5, steps=24, precision=0, guess=2, **ODD),
        # a scan with the production couplings
        dict(name="scan_production_8", call="scan", batch=8, steps=2, precision=0, guess=0, **PRODUCTION),
        # a program that stays with the assembled matrices
        dict(name="assembled_middle", call="assembled", **MIDDLE),
        # what is printed about a state at an output
        dict(name="populations_middle", call="populations", **MIDDLE),
        # one training batch of the learned guess
        dict(name="guess_grad_256", call="guess_grad", rows=256),
    ]


def _size(case):
    """(row blocks, radial functions) of a configuration."""
    nk, nmu = case["nkappa"], case["nmu"]
    kappas = [s * k for k in range(1, nk + 1) for s in (1, -1)]
    if nk == 1:
        kappas = [-1, 1]
    rows = sum(2 * min(abs(k), nmu) if nmu else 2 * abs(k) for k in kappas)
    return rows, 2 * (case["nsplines"] + 5)


def draw(rng):
    call = rng.choice(["apply", "apply", "precondition", "run", "run", "run", "scan", "scan", "scan", "assembled",
                       "populations", "guess_grad"])
    if call == "guess_grad":
        return dict(call=call, rows=16 * rng.randint(4, 64))
    # box resolution, angular momenta and multipoles of a calculation, from the dipole size to the production size
    big = {"assembled": 100, "populations": 120, "scan": 160}.get(call, 250)
    nk = rng.randint(3, {"assembled": 8, "populations": 8, "scan": 12}.get(call, 16))
    nmu = rng.choice([0, max(2, nk // 2)]) if nk <= 8 else nk // 2
    case = dict(call=call, nsplines=int(round(math.exp(rng.uniform(math.log(20), math.log(big))))), nkappa=nk,
                nmu=nmu, nl=rng.randint(1, min(8, nk)) if call != "assembled" else rng.randint(1, 4),
                cycles=rng.randint(1, 15), per_cycle=rng.randint(200, 600))
    if call in ("run", "scan"):
        n = _size(case)[0] * _size(case)[1]
        most = 16 * 204000  # entries times steps of the largest listed run
        if call == "scan":
            case["batch"] = max(2, min(int(round(math.exp(rng.uniform(math.log(2), math.log(64))))), most // (4 * n)))
        case["steps"] = max(2, min(rng.randint(4, 60), most // (n * case.get("batch", 1))))
        case["precision"] = int(rng.random() < 0.25)
        case["guess"] = rng.choice([0, 0, 0, 1, 2, 3])
    return case


# ---- the couplings and the models of this process ----------------------------------------------------------------
_dirs, _models = {}, {}


def _couplings(case):
    key = tuple(case[k] for k in ("nsplines", "nkappa", "nmu", "nl", "cycles"))
    if key not in _dirs:
        if not _dirs:
            _dirs[None] = tempfile.mkdtemp(prefix="couplings_")
            atexit.register(shutil.rmtree, _dirs[None], ignore_errors=True)
        d = os.path.join(_dirs[None], "_".join(map(str, key)))
        generate(d, nsplines=case["nsplines"], nkappa=case["nkappa"], nmu=case["nmu"], nl=case["nl"], rbox=RBOX, Z=1,
                 intensity=10, omega=OMEGA, cycles=case["cycles"])
        _dirs[key] = d
    return _dirs[key]


def _dt(case):
    return 2 * math.pi / OMEGA / case["per_cycle"]


def _model(case):
    """The model of a configuration with what a program sets up once."""
    key = tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "steps", "rows")))
    if key not in _models:
        if len(_models) > 12:
            _models.pop(next(iter(_models))).close()
        if case["call"] == "guess_grad":
            small = dict(DIPOLE)
            p = gade.Propagator(_couplings(small), small["nl"], _dt(small))
            p.lg_set_norm(np.full(gade.LG_IN, 0.5, np.float32), np.full(gade.LG_IN, 2.0, np.float32))
            p.lg_set_params(_network())
        else:
            p = gade.Propagator(_couplings(case), case["nl"], _dt(case), batch=case.get("batch", 1))
            if case.get("precision"):
                p.set_param("precision", 1)
            if case.get("guess"):
                p.set_param("guess_order", case["guess"])
            if case["call"] in ("precondition", "run", "scan"):
                gade.check(gade.lib().gade_precond_setup(p.ptr))
            if case["call"] == "populations":
                p.eig_values()
        _models[key] = p
    return _models[key]


def _network():
    """Weights of a trained size: He-normal layers, a small output layer (float32, the library's flat order)."""
    rng = np.random.default_rng(7)
    out = []
    for k, (fi, fo) in enumerate(_LAYERS):
        out.append((rng.standard_normal(fo * fi) * math.sqrt((2.0 if k < 3 else 0.02) / fi)).astype(np.float32))
        out.append((0.05 * rng.standard_normal(fo)).astype(np.float32))
    return np.concatenate(out)


_LAYERS = [(gade.LG_IN, gade.LG_HIDDEN), (gade.LG_HIDDEN, gade.LG_HIDDEN), (gade.LG_HIDDEN, gade.LG_HIDDEN),
           (gade.LG_HIDDEN, gade.LG_OUT)]


class _Vec:
    """A tensor as the library takes it: by its device pointer."""

    def __init__(self, t):
        self.t, self.ptr = t, t.data_ptr()


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


# ---- inputs -----------------------------------------------------------------------------------------------------
def _states(case, seed, batch):
    """batch states in the middle of a pulse [batch][rows][radial] (host): the ground state and wave packets that
    the field has put into the other blocks, fewer the higher the angular momentum."""
    psi0, _ = gade.read_psi0(_couplings(case), _size(case)[0] * _size(case)[1])
    nblk, n = _size(case)
    rng = np.random.default_rng(seed)
    kap = np.abs(_kappas(case))
    x = np.linspace(0.0, 1.0, n // 2)
    c = rng.uniform(0.05, 0.6, (batch, nblk, 1))
    k = rng.uniform(-0.2, 0.2, (batch, nblk, 1)) * (n // 2)
    a = 0.3 * (rng.standard_normal((batch, nblk, 1)) + 1j * rng.standard_normal((batch, nblk, 1))) / kap[:, None] ** 2
    packet = a * np.exp(-((x - c) / 0.12) ** 2 + 1j * k * x)
    psi = np.tile(psi0.reshape(1, nblk, n), (batch, 1, 1))
    psi[:, :, :n // 2] += packet
    psi[:, :, n // 2:] += packet * rng.uniform(-1, 1, (batch, nblk, 1)) / (2 * SOL)
    return psi


def _pulses(case, seed, batch):
    """(E0, omega, cycles, cep) of each pulse; a single run has the reference's carrier phase."""
    rng = np.random.default_rng(seed + 1)
    p = np.zeros((batch, 4))
    p[:, 0] = rng.uniform(5.0, 15.0, batch)
    p[:, 1] = rng.uniform(45.0, 55.0, batch)
    p[:, 2] = case["cycles"]
    if case["call"] == "scan":
        p[:, 3] = rng.uniform(0.0, 2 * math.pi, batch)
    return p


def _start(case):
    """Time at which the steps begin: shortly before the middle of the envelope."""
    return 0.4 * case["cycles"] * 2 * math.pi / OMEGA


def _f(pulse, t):
    """f_alpha(t) of a pulse, alpha = 0..5 (the sin^2 envelope as three carriers)."""
    e0, w, cycles, cep = (float(v) for v in pulse)
    d, ph = w / cycles, -math.pi / 2 + cep
    return np.array([-e0 / (4 * w) * math.cos(ph + t * (d + w)), -e0 / (4 * w) * math.sin(ph + t * (d + w)),
                     -e0 / (4 * w) * math.cos(-ph + t * (d - w)), e0 / (4 * w) * math.sin(-ph + t * (d - w)),
                     e0 / (2 * w) * math.cos(ph + t * w), e0 / (2 * w) * math.sin(ph + t * w)], np.complex128)


def _samples(case, seed):
    """Training samples [rows][LG_SAMPLE]: inputs, then the quadratic form of a guess error in the span of the
    differences and the basis, from vectors of a small space."""
    M, n, npod = case["rows"], 160, gade.LG_POD
    g = torch.Generator().manual_seed(seed)

    def cn(*shape):
        return torch.complex(torch.randn(*shape, generator=g, dtype=torch.float64),
                             torch.randn(*shape, generator=g, dtype=torch.float64))

    U = torch.linalg.qr(cn(n, npod))[0]
    D = cn(M, n, 6)
    D = D / torch.linalg.vector_norm(D, dim=1, keepdim=True)
    e = 0.3 * cn(M, n) / math.sqrt(n)
    x = 2 * torch.randn(M, gade.LG_IN, generator=g, dtype=torch.float64) + 1
    G = (D.mH @ D).real
    a = (D.mH @ e[:, :, None]).real[:, :, 0]
    P = U.mH @ D
    q = e @ U.conj()
    s = torch.zeros(M, gade.LG_SAMPLE, dtype=torch.float64)
    parts = [x, G.reshape(M, -1), a, torch.view_as_real(P).reshape(M, -1), torch.view_as_real(q).reshape(M, -1),
             (e.abs() ** 2).sum(1, keepdim=True), torch.ones(M, 1, dtype=torch.float64)]
    s[:, :sum(p.shape[1] for p in parts)] = torch.cat(parts, 1)
    return s.float()


def prepare(case, seed):
    p = _model(case)
    dev = _device()
    if case["call"] == "guess_grad":
        M = case["rows"]
        return dict(case=case, p=p, samples=_Vec(_samples(case, seed).to(dev).contiguous()),
                    idx=_Vec(torch.randperm(M, generator=torch.Generator().manual_seed(seed)).to(torch.int32).to(dev)),
                    grad=_Vec(torch.zeros(gade.LG_PARAMS, dtype=torch.float32, device=dev)))
    batch = case.get("batch", 1)
    psi = torch.from_numpy(_states(case, seed, batch).reshape(-1)).to(dev)
    s = dict(case=case, p=p, x=_Vec(psi), y=_Vec(torch.zeros_like(psi)))
    pulses = _pulses(case, seed, batch)
    if case["call"] in ("apply", "assembled"):
        s["f"] = _f(pulses[0], _start(case))
    if case["call"] in ("run", "scan"):
        s["pulses"] = pulses
    return s


def run(s):
    case, p, call = s["case"], s["p"], s["case"]["call"]
    if call == "apply":
        p.set_time(s["f"])
        p.apply(s["x"], s["y"])
        return s["y"].t
    if call == "precondition":
        p.psolve(s["x"], s["y"])
        return s["y"].t
    if call == "run":
        s["y"].t.copy_(s["x"].t)
        e0, omega, cycles, _ = s["pulses"][0]
        p.reset_workspace()
        p.cn_run(s["y"], e0, omega, cycles, case["steps"], t0=_start(case), tol=TOL, timing=False)
        return s["y"].t
    if call == "scan":
        s["y"].t.copy_(s["x"].t)
        p.reset_workspace()
        p.cn_run_batch(s["y"], s["pulses"], case["steps"], t0=_start(case), tol=TOL)
        return s["y"].t
    if call == "assembled":
        p.set_time(s["f"])
        p.assembled_timedep()
        p.assembled_spmv(s["x"], s["y"], alpha=1.0, beta=0.0, with_S=True)
        return s["y"].t
    if call == "populations":
        return p.populations(s["x"], per_block=True)
    loss = p.lg_grad(s["samples"], s["idx"], case["rows"], s["grad"])
    return {"loss": loss, "grad": s["grad"].t}


# ---- what a pass cannot do without ------------------------------------------------------------------------------
def work(case):
    if case["call"] == "guess_grad":
        w = sum(fi * fo for fi, fo in _LAYERS)
        return {"bytes": 4 * (case["rows"] * gade.LG_SAMPLE + 2 * gade.LG_PARAMS), "flops": 6.0 * case["rows"] * w}
    nblk, n = _size(case)
    ns, nl = n // 2, case["nl"]
    N = float(nblk * n)
    nnz_b = 4 * sum(min(ns - 1, i + 7) - max(0, i - 7) + 1 for i in range(ns))
    lists = _coupled(case)
    # one operator product: the angular couplings with and without kappa (real factors), four banded products per
    # multipole (real factors) and the complex stationary operator
    apply_flops = 4.0 * lists * 2 * n + 4.0 * nblk * nnz_b * 4 * nl + 8.0 * nblk * nnz_b
    coupling_bytes = 8.0 * 24 * nl * nnz_b
    nk = 2 * case["nkappa"]
    solve_flops = 8.0 * nblk * nnz_b * 2
    call, B, steps = case["call"], case.get("batch", 1), case.get("steps", 1)
    if call == "apply":
        return {"bytes": coupling_bytes + 8.0 * 7 * nnz_b + 32 * N, "flops": apply_flops}
    if call == "precondition":
        return {"bytes": 16.0 * nk * nnz_b + 32 * N, "flops": solve_flops}
    if call in ("run", "scan"):
        # per step the right-hand side, A x0 and one body: four products and two solves
        return {"bytes": coupling_bytes + 8.0 * 7 * nnz_b + 32 * N * B,
                "flops": B * steps * (4 * apply_flops + 2 * solve_flops)}
    if call == "assembled":
        full = float(len(_pattern(case)[0])) * nnz_b
        return {"bytes": coupling_bytes + 16 * full + 20 * full + 32 * N, "flops": 8.0 * full + 4.0 * lists * 4 * nnz_b}
    return {"bytes": 16 * N + 8.0 * nk * n * n, "flops": 4.0 * N * n}


# ---- the same in 64 bits, from the files alone ------------------------------------------------------------------
def _csr(path):
    """(rows, columns, values, trailer) of a coupling file: int32 n, nnz, Ap, Ai, complex128 values."""
    raw = open(path, "rb").read()
    n, nnz = struct.unpack_from("ii", raw)
    ap = np.frombuffer(raw, np.int32, n + 1, 8)
    ai = np.frombuffer(raw, np.int32, nnz, 8 + 4 * (n + 1))
    off = 8 + 4 * (n + 1 + nnz)
    return np.repeat(np.arange(n), np.diff(ap)), ai, np.frombuffer(raw, np.complex128, nnz, off), raw[off + 16 * nnz:], n


def _pattern(case):
    """(block rows, block columns, original index of each block) of H.csr."""
    rows, cols, _, rest, n = _csr(os.path.join(_couplings(case), "H.csr"))
    return rows, cols, np.frombuffer(rest, np.int32, n)


def _kappas(case):
    """kappa of each block: shell k holds 4k states, first kappa = -k, then kappa = k."""
    out = []
    for i in _pattern(case)[2]:
        k = 1
        while i >= 2 * k * (k + 1):
            k += 1
        out.append(-k if i - 2 * k * (k - 1) < 2 * k else k)
    return np.array(out)


def _angular(case):
    """H0l, H1l between the kept blocks, [nl][2][rows][rows]; a pair that H.csr leaves out does not couple."""
    rows, cols, perm = _pattern(case)
    kept = np.zeros((len(perm), len(perm)), bool)
    kept[rows, cols] = True
    out = np.zeros((case["nl"], 2, len(perm), len(perm)), np.complex128)
    for l in range(case["nl"]):
        for j in (0, 1):
            r, c, v, _, n = _csr(os.path.join(_couplings(case), "H%dl%d.csr" % (j, l)))
            m = np.zeros((n, n), np.complex128)
            m[r, c] = v
            out[l, j] = m[np.ix_(perm, perm)] * kept
    return out


_counts = {}


def _coupled(case):
    key = tuple(case[k] for k in ("nkappa", "nmu", "nl"))
    if key not in _counts:
        _counts[key] = int(np.count_nonzero(_angular(case)))
    return _counts[key]


def _dense(case, name, dev):
    r, c, v, _, n = _csr(os.path.join(_couplings(case), name + ".csr"))
    m = np.zeros((n, n), np.complex128)
    m[r, c] = v
    return torch.from_numpy(m).to(dev)


class _Exact:
    """S, H0 and H(t) of a configuration as dense matrices (complex128)."""

    def __init__(self, case):
        dev = _device()
        self.dev, self.nl, self.dt = dev, case["nl"], _dt(case)
        self.kap = torch.from_numpy(_kappas(case).astype(np.float64)).to(dev)
        self.kq, self.q = torch.unique(self.kap, return_inverse=True)
        s = [_dense(case, "s%d" % i, dev) for i in range(3)]
        h = [_dense(case, "h0%d" % i, dev) for i in range(4)]
        self.S = torch.stack([s[0] + k * s[1] + k * k * s[2] for k in self.kq.tolist()])
        self.H0 = torch.stack([h[0] + k * h[1] + k * k * h[2] + k ** 3 * h[3] for k in self.kq.tolist()])
        if case["call"] not in ("precondition", "populations"):
            self.ang = torch.from_numpy(_angular(case)).to(dev)
            self.g = [[torch.stack([_dense(case, "g%da%dl%d" % (n, a, l), dev) for a in range(l % 2 == 0, 6, 2)])
                       for n in range(4)] for l in range(self.nl)]

    def rows(self, mats, x):
        """mats[kappa of the row] applied to every row of x [B][rows][n]."""
        out = torch.empty_like(x)
        for q in range(len(self.kq)):
            at = torch.nonzero(self.q == q)[:, 0]
            out[:, at] = x[:, at] @ mats[q].T
        return out

    def set_time(self, f):
        """f [B][6]: the interaction matrices of every instance."""
        c = torch.from_numpy(1j * self.dt / 2 * SOL * np.asarray(f)).to(self.dev)
        self.G = []
        for l in range(self.nl):
            w = c[:, (l % 2 == 0)::2]
            gs = [torch.einsum("ba,aij->bij", w, g) for g in self.g[l]]
            gt = [torch.einsum("ba,aij->bij", w, g.conj().transpose(1, 2)) for g in self.g[l]]
            self.G.append((gs, gt))

    def interaction(self, x):
        k = self.kap[:, None].to(torch.complex128)
        y = torch.zeros_like(x)
        for l in range(self.nl):
            gs, gt = self.G[l]
            z0, z2 = self.ang[l, 0] @ x, self.ang[l, 0] @ (k * x)
            w0, w1 = self.ang[l, 1] @ x, self.ang[l, 1] @ (k * x)
            for v, a, b in ((z0, gs[0], gs[1]), (z2, gs[2], gs[3]), (w0, gt[0], gt[2]), (w1, gt[1], gt[3])):
                y += v @ a.transpose(1, 2) + k * (v @ b.transpose(1, 2))
        return y

    def apply(self, x, sign):
        """(S + sign H) x."""
        return self.rows(self.S + sign * 1j * self.dt / 2 * self.H0, x) + sign * self.interaction(x)

    def inverse(self):
        if not hasattr(self, "Pinv"):
            self.Pinv = torch.linalg.inv((self.S + 1j * self.dt / 2 * self.H0).cpu()).to(self.dev)
            # one Newton step takes the inverse's own rounding out
            eye = torch.eye(self.S.shape[1], dtype=torch.complex128, device=self.dev)
            self.Pinv = self.Pinv @ (2 * eye - (self.S + 1j * self.dt / 2 * self.H0) @ self.Pinv)
        return self.Pinv

    def precondition(self, b):
        x = self.rows(self.inverse(), b)
        P = self.S + 1j * self.dt / 2 * self.H0
        for _ in range(2):
            x = x + self.rows(self.Pinv, b - self.rows(P, x))
        return x

    def step(self, x):
        """x_{n+1} of (S + H) x_{n+1} = (S - H) x_n, by iteration on the block-diagonal part."""
        b, best = self.apply(x, -1), math.inf
        for _ in range(60):
            r = b - self.apply(x, 1)
            size = float(torch.linalg.vector_norm(r) / torch.linalg.vector_norm(b))
            if size < 1e-15 or size > 0.7 * best and size < 1e-13:
                return x
            best = min(best, size)
            x = x + self.rows(self.inverse(), r)
        return None


_exacts = {}


def _exact_of(case):
    key = tuple(sorted((k, v) for k, v in case.items() if k in ("nsplines", "nkappa", "nmu", "nl", "cycles", "per_cycle")))
    key += (case["call"] in ("precondition", "populations"),)
    if key not in _exacts:
        _exacts.clear()
        _exacts[key] = _Exact(case)
    return _exacts[key]


def exact(case, seed):
    call = case["call"]
    if call == "guess_grad":
        return _exact_grad(case, seed)
    e, batch = _exact_of(case), case.get("batch", 1)
    x = torch.from_numpy(_states(case, seed, batch)).to(e.dev)
    pulses = _pulses(case, seed, batch)
    if call in ("apply", "assembled"):
        e.set_time([_f(pulses[0], _start(case))])
        return e.apply(x, 1).reshape(-1)
    if call == "precondition":
        return e.precondition(x).reshape(-1)
    if call in ("run", "scan"):
        t = _start(case)
        for _ in range(case["steps"]):
            t += e.dt
            e.set_time([_f(p, t) for p in pulses])
            x = e.step(x)
            if x is None:
                return None
        return x.reshape(-1)
    w = e.rows(e.S, x)[0]
    out = torch.zeros(len(e.kap), 4, dtype=torch.float64, device=e.dev)
    for q in range(len(e.kq)):
        L = torch.linalg.cholesky(e.S[q].real.cpu())
        A = torch.linalg.solve_triangular(L, e.H0[q].real.cpu(), upper=False)
        A = torch.linalg.solve_triangular(L, A.T.contiguous(), upper=False)
        E, V = torch.linalg.eigh((A + A.T) / 2)
        V = torch.linalg.solve_triangular(L.T.contiguous(), V, upper=True).to(e.dev).to(torch.complex128)
        E = E.to(e.dev)
        at = torch.nonzero(e.q == q)[:, 0]
        pop = (w[at] @ V.conj()).abs() ** 2
        out[at, 0] = pop[:, E < -SOL ** 2].sum(1)
        out[at, 1] = pop[:, (E >= -SOL ** 2) & (E < 0)].sum(1)
        out[at, 2] = pop[:, E >= 0].sum(1)
        out[at, 3] = (x[0][at].conj() * w[at]).sum(1).real
    out = out.cpu().numpy()
    return dict(norm=float(out[:, 3].sum()), bound=float(out[:, 1].sum()), ionised=float(out[:, 2].sum()), per_block=out)


def _exact_grad(case, seed):
    s = _samples(case, seed).double()
    order = torch.randperm(case["rows"], generator=torch.Generator().manual_seed(seed))
    s = s[order]
    flat = torch.from_numpy(_network()).double().requires_grad_()
    a = (s[:, :gade.LG_IN] - 0.5) / 2.0
    a = torch.where(torch.arange(gade.LG_IN) < gade.LG_FEATURES, a, torch.zeros(()).double())
    o = 0
    for k, (fi, fo) in enumerate(_LAYERS):
        a = a @ flat[o:o + fo * fi].reshape(fo, fi).T + flat[o + fo * fi:o + fo * fi + fo]
        o += fo * fi + fo
        if k < 3:
            a = torch.nn.functional.gelu(a)
    npod, o = gade.LG_POD, gade.LG_IN
    G = s[:, o:o + 36].reshape(-1, 6, 6)
    lin = s[:, o + 36:o + 42]
    P = torch.view_as_complex(s[:, o + 42:o + 42 + 12 * npod].reshape(-1, npod, 6, 2).contiguous())
    q = torch.view_as_complex(s[:, o + 42 + 12 * npod:o + 42 + 14 * npod].reshape(-1, npod, 2).contiguous())
    beta = s[:, o + 42 + 14 * npod]
    w = a[:, :6]
    c = torch.view_as_complex(a[:, 6:6 + 2 * npod].reshape(-1, npod, 2).contiguous())
    Pw = (P @ w[:, :, None].to(torch.complex128))[:, :, 0]
    loss = (beta - 2 * (w * lin).sum(1) + (w[:, None, :] @ G @ w[:, :, None])[:, 0, 0]
            - 2 * (c.conj() * q).sum(1).real + (c.abs() ** 2).sum(1) + 2 * (c.conj() * Pw).sum(1).real) / beta
    loss = loss.mean()
    loss.backward()
    return {"loss": loss.item(), "grad": flat.grad.detach()}
