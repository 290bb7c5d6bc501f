"""Measured workloads of phi_amd: what a user has the integrator do, over the
range of sizes it takes, each through the public entry points.

Kinds of case (key "kind"):
  launch     HierarchyIntegrator: create, Launch(), density_matrix(), state():
             the whole call of the `phi` program for a small open system
  rk4        Context.rk4_history on one hierarchy: FP64 and FP32 bulk, from a
             few sites to systems above the matrix-core limit of 32 sites
  rkf45      Context.rkf45_attempt / rkf45_accept: an adaptive controller's loop
  ensemble   Ensemble.rk4_history: static disorder, uneven depths
  steady     Context.set_state + steady_state / steady_state_l
  closure    Ensemble with a learned truncation closure attached
  train      Mlp.set_params + train + get_params of the closure network
  bath       Context.rk4_history with full coupling operators
  rhs        Context.rhs: the batched Get for a caller with a loop of its own
"""

import math

import numpy as np
import torch

import phi_amd as P

HBAR, KB = 5.3088354, 0.6950344  # cm^-1 ps, cm^-1 / K (PHI's defaults)


# --- Cases -------------------------------------------------------------------------

def _case(name, kind, **kw):
    c = {"kind": kind, "sites": 7, "lh": 9, "terms": 1, "lam": 35.0, "gam": 20.0, "temp": 77.0,
         "precision": "fp64", "steps": 1, "every": 10, "members": 0, "autotune": False, "ell": 0,
         "rows": 0, "batch": 0, "epochs": 0, "state": False}
    if name:
        c["name"] = name
    c.update(kw)
    return c


def listed():
    return [
        # The dimer of phi_amd/configs/c1.prm (495 nodes of 2x2) integrated to
        # 1 ps by the whole program call: the smallest job, all latency.
        _case("dimer_launch_fp64", "launch", sites=2, lh=9, terms=2, temp=300.0, steps=1000),
        # The 7-site exciton of configs/c2.prm alone (6435 nodes of 7x7),
        # plain FP64: 1 ps of dynamics with an output line every 10 fs, then
        # the whole state (for a restart or further analysis).
        _case("site7_rk4_fp64", "rk4", steps=1000, state=True),
        # The 24-site ring of configs/c3.prm (20475 nodes of 24x24), FP32 bulk.
        _case("ring24_rk4_fp32", "rk4", sites=24, lh=5, lam=50.0, gam=10.0, temp=300.0,
              precision="fp32", steps=100),
        # The same ring under an adaptive controller, plain FP64.
        _case("ring24_rkf45_fp64", "rkf45", sites=24, lh=5, lam=50.0, gam=10.0, temp=300.0,
              steps=16),
        # A system wider than the matrix-core kernels take (34 sites, 630
        # nodes): the one-shot kernels.
        _case("site34_rk4_fp64", "rk4", sites=34, lh=3, lam=50.0, gam=10.0, temp=300.0, steps=40),
        # bench.py's headline ensemble: 512 realisations of the 7-site system,
        # depths 4..8, FP32 bulk, autotuned once as there.
        _case("ensemble512_fp32", "ensemble", members=512, precision="fp32", steps=30,
              autotune=True),
        # A modest FP64 ensemble with a Matsubara term (two modes per site):
        # 96 four-site realisations of uneven depth, default launch shape.
        _case("ensemble96_fp64", "ensemble", sites=4, lh=6, terms=2, members=96, steps=200),
        # Steady state of the 7-site system from the initial state by PHI's
        # `bicgstab` word (BiCGSTAB(2)), to residual 1e-10.
        _case("site7_steady_l2", "steady", ell=2),
        # The closure study's evaluation: 256 Hamiltonians at depth 4 + closure.
        _case("closure256_fp32", "closure", lh=5, members=256, precision="fp32", steps=50),
        # Training the closure network (105 -> 256 -> 256 -> 686), batch 512.
        _case("train_batch512", "train", lh=5, rows=16384, batch=512, epochs=3),
        # Full (non-projector) coupling operators, 7 sites, 792 nodes.
        _case("bath_full_fp64", "bath", lh=6, steps=40, state=True),
        # One batched Get from host arrays, 7 sites at depth 5 (792 nodes).
        _case("rhs_host_fp64", "rhs", lh=6),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def nodes(modes, lh):
        return math.comb(modes + lh - 1, lh - 1)

    def sized(sites, terms, most, lh_min=2, lh_max=12):
        ok = [l for l in range(lh_min, lh_max + 1) if nodes(sites * terms, l) * sites ** 2 <= most]
        return rng.choice(ok or [lh_min])

    kind = rng.choice(["launch", "rk4", "rk4", "rkf45", "ensemble", "ensemble", "steady",
                       "closure", "train", "bath", "rhs"])
    base = {"lam": round(rng.uniform(5.0, 60.0), 2), "gam": round(rng.uniform(5.0, 25.0), 2),
            "temp": round(rng.uniform(70.0, 320.0), 1)}
    prec = rng.choice(["fp64", "fp32"])
    if kind == "launch":
        n, t = rng.randint(2, 5), rng.randint(1, 2)
        return _case(None, kind, sites=n, terms=t, lh=sized(n, t, 20000, 3),
                     steps=log_int(100, 2000), precision=prec, **base)
    if kind == "rk4":
        n = log_int(2, 36)
        n = 24 if 24 < n < 33 else n  # FP64 tiles of 27..32 sites exceed the kernels' LDS
        t = rng.randint(1, 2) if n <= 16 else 1
        lh = sized(n, t, 8_000_000, 2 if n > 16 else 3)
        return _case(None, kind, sites=n, terms=t, lh=lh, precision=prec,
                     steps=log_int(12, 120), every=rng.randint(1, 12),
                     state=nodes(n * t, lh) * n * n <= 100_000, **base)
    if kind == "rkf45":
        n = log_int(2, 24)
        return _case(None, kind, sites=n, lh=sized(n, 1, 6_000_000, 3),
                     steps=rng.randint(5, 16), **base)
    if kind == "ensemble":
        n, t = rng.randint(2, 10), rng.randint(1, 2)
        lh = sized(n, t, 300_000, 4, 9)
        m = max(3, min(log_int(8, 400), 30_000_000 // (nodes(n * t, lh) * n * n)))
        return _case(None, kind, sites=n, terms=t, lh=lh, members=m, precision=prec,
                     steps=log_int(12, 90), every=rng.randint(2, 20), **base)
    if kind == "steady":
        n = rng.randint(3, 7)
        return _case(None, kind, sites=n, lh=sized(n, 1, 350_000, 4, 9),
                     ell=rng.choice([0, 1, 2, 2, 4]), lam=35.0, gam=20.0,
                     temp=round(rng.uniform(77.0, 300.0), 1))
    if kind == "closure":
        n = rng.randint(4, 7)
        return _case(None, kind, sites=n, lh=rng.randint(3, 5), members=log_int(16, 256),
                     precision=prec, steps=log_int(12, 50), lam=35.0, gam=20.0, temp=77.0)
    if kind == "train":
        return _case(None, kind, sites=rng.randint(4, 7), lh=5, rows=log_int(3000, 16384),
                     batch=rng.choice([128, 256, 300, 512, 777, 1024]), epochs=rng.randint(1, 3))
    if kind == "bath":
        n = rng.randint(2, 7)
        return _case(None, kind, sites=n, lh=sized(n, 1, 40_000, 3, 8), steps=log_int(10, 40),
                     state=True, **base)
    n = log_int(2, 12)
    return _case(None, "rhs", sites=n, lh=sized(n, 1, 120_000, 3), **base)


# --- Inputs --------------------------------------------------------------------------

def _rng(case, seed):
    return np.random.default_rng([int(seed) & 0x7FFFFFFF, case["sites"], case["lh"]])


def _hamiltonian(case, rng):
    """Site energies and couplings in the ranges of phi_amd/configs (an
    alternating ring for the wide systems)."""
    n = case["sites"]
    H = np.diag(rng.uniform(12200.0, 12600.0, size=n))
    if n < 12:
        J = np.clip(rng.normal(0.0, 40.0, size=(n, n)), -120.0, 120.0)
        iu = np.triu_indices(n, 1)
        H[iu] = J[iu]
        H[(iu[1], iu[0])] = J[iu]
    else:
        for i in range(n):
            j, k = (i + 1) % n, (i + 2) % n
            H[i, j] = H[j, i] = 300.0 if i % 2 == 0 else 230.0
            H[i, k] = H[k, i] = -30.0
    return H


def _rho0(n):
    r = np.zeros((n, n), dtype=complex)
    r[0, 0] = 1.0
    return r


def _params(case, H, method="rk4", lh=None):
    n = case["sites"]
    return P.params_from_problem(
        H, _rho0(n), gamma=[case["gam"]] * n, lambda_=[case["lam"]] * n,
        temperature=case["temp"], lh=lh or case["lh"], num_terms=case["terms"],
        dt=0.001, t_end=0.001 * case["steps"] - 0.0005, method=method,
        precision=case["precision"])


def _depths(case):
    """PHI depths of the members: uneven, the same for every seed."""
    r = np.random.default_rng(case["members"])
    if case["kind"] == "closure":
        return [case["lh"]] * case["members"]
    d = r.integers(max(2, case["lh"] - 4), case["lh"] + 1, size=case["members"])
    d[0] = case["lh"]
    return [int(v) for v in d]


def _members(case, seed):
    rng = _rng(case, seed)
    H = _hamiltonian(case, rng)
    disorder = rng.normal(0.0, 100.0, size=(case["members"], case["sites"]))
    return np.array([H + np.diag(d) for d in disorder])


def _net_sizes(case):
    n = case["sites"]
    return 2 * n * n + n * case["terms"], 256, 2 * n * n * n * case["terms"]


def _net_params(case, seed):
    rng = np.random.default_rng([int(seed) & 0x7FFFFFFF, 77])
    i, h, o = _net_sizes(case)
    parts = []
    for a, b, s in ((i, h, 1.0), (h, h, 1.0), (h, o, 0.1)):
        parts += [rng.standard_normal((b, a)).reshape(-1) * math.sqrt(2.0 / a) * s, np.zeros(b)]
    return np.concatenate(parts).astype(np.float32)


def _bath_ops(case, rng):
    """Site projectors with symmetric off-diagonal parts, one per bath."""
    n = case["sites"]
    F = np.zeros((n, n, n))
    for m in range(n):
        g = 0.1 * rng.standard_normal((n, n))
        F[m] = 0.5 * (g + g.T)
        F[m, m, m] += 1.0
    return F


def _training_rows(case, seed):
    """Rows with the closure's input ranges (|entries| <= 1, occupations over
    the depth) and targets a smooth function of them."""
    rng = np.random.default_rng([int(seed) & 0x7FFFFFFF, 5])
    i, _, o = _net_sizes(case)
    d = case["sites"] * case["terms"]
    X = rng.uniform(-1.0, 1.0, size=(case["rows"], i)).astype(np.float32)
    X[:, i - d:] = rng.integers(0, case["lh"], size=(case["rows"], d)) / (case["lh"] - 1.0)
    A = rng.standard_normal((i, o)).astype(np.float32) / math.sqrt(i)
    return X, (0.3 * np.tanh(X @ A)).astype(np.float32)


def _rkf45_coefs(dt):
    b = [2. / 9., 1. / 12., 1. / 4., 69. / 128., -243. / 128., 135. / 64., -17. / 12., 27. / 4.,
         -27. / 5., 16. / 15., 65. / 432., -5. / 16., 13. / 16., 4. / 27., 5. / 144.]
    c4 = [1. / 9., 9. / 20., 16. / 45., 1. / 12.]
    c5 = [47. / 450., 12. / 25., 32. / 225., 1. / 30., 6. / 25.]
    return dt * np.array(b + c4 + c5)


def _rhs_input(case, seed):
    """Hermitian blocks that decay over the hierarchy, as ADOs do."""
    rng = _rng(case, seed + 1)
    n = case["sites"]
    k = math.comb(n * case["terms"] + case["lh"] - 1, case["lh"] - 1)
    x = rng.standard_normal((k, n, n)) + 1j * rng.standard_normal((k, n, n))
    x = 0.5 * (x + x.conj().transpose(0, 2, 1))
    return x / (1.0 + np.arange(k))[:, None, None] ** 0.5


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "dt": 0.001}
    if kind == "train":
        i, h, o = _net_sizes(case)
        s["X"], s["T"] = _training_rows(case, seed)
        s["flat"] = _net_params(case, seed)
        s["net"] = P.Mlp(i, h, o, max_batch=max(case["batch"], 8192))
        return s
    if kind in ("ensemble", "closure"):
        Hs = _members(case, seed)
        p = _params(case, Hs[0])
        ens = P.Ensemble(p, Hs, _depths(case), precision=case["precision"])
        if kind == "closure":
            i, h, o = _net_sizes(case)
            s["net"] = P.Mlp(i, h, o, max_batch=8192)
            s["net"].set_params(_net_params(case, seed))
            ens.attach_closure(s["net"])
        if case["autotune"]:
            ens.autotune(s["dt"], steps=3)
        s["ctx"] = ens
        return s
    rng = _rng(case, seed)
    H = _hamiltonian(case, rng)
    p = _params(case, H)
    if kind == "launch":
        s["params"] = p
        return s
    if kind == "bath":
        ops = _bath_ops(case, rng)
        p.set_int("is_full_bath_coupling", 1)
        p.set_array("bath_coupling_op", np.ascontiguousarray(ops.transpose(0, 2, 1)).reshape(-1))
        if p.fix("rk4") != 0:
            raise RuntimeError("bath parameters refused")
    s["ctx"] = ctx = P.Context(p, precision=case["precision"])
    if kind in ("rk4", "rkf45", "bath", "steady"):
        x0 = np.zeros((ctx.num_nodes, case["sites"], case["sites"]), dtype=complex)
        x0[0] = _rho0(case["sites"])
        if kind == "steady":
            s["x0"] = x0
        else:
            ctx.set_state(x0)
    if kind == "rkf45":
        s["coefs"] = _rkf45_coefs(s["dt"])
    if kind == "rhs":
        s["x"] = _rhs_input(case, seed)
    return s


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "launch":
        it = P.HierarchyIntegrator(s["params"])
        it.Launch()
        return [it.density_matrix(), it.state()]
    if kind == "train":
        s["net"].set_params(s["flat"])
        losses = s["net"].train(s["X"], s["T"], batch=case["batch"], epochs=case["epochs"],
                                lr=1e-3, lr_final=1e-5, seed=1)
        return [losses, s["net"].get_params()]
    ctx = s["ctx"]
    if kind in ("rk4", "bath"):
        return [ctx.rk4_history(case["steps"], s["dt"], case["every"]),
                ctx.state() if case["state"] else ctx.rho0()]
    if kind in ("ensemble", "closure"):
        return [ctx.rk4_history(case["steps"], s["dt"], case["every"]), ctx.member_rho0()]
    if kind == "rkf45":
        errs = []
        for _ in range(case["steps"]):
            errs.append(ctx.rkf45_attempt(s["coefs"]))
            ctx.rkf45_accept()
        return [np.array(errs), ctx.rho0()]
    if kind == "steady":
        ctx.set_state(s["x0"])
        if case["ell"] == 0:
            rc, _, _ = ctx.steady_state(1e-10, 20000)
        else:
            rc, _, _ = ctx.steady_state_l(case["ell"], 1e-10, 20000)
        return [rc, ctx.rho0()]
    return [ctx.rhs(s["x"])]


# --- What a pass cannot do without --------------------------------------------------

def work(case):
    kind, n, d = case["kind"], case["sites"], case["sites"] * case["terms"]
    if kind == "train":
        i, h, o = _net_sizes(case)
        weights = i * h + h * h + h * o
        batches = case["rows"] // case["batch"]
        rows = batches * case["batch"]
        # each row read once an epoch; parameters, both Adam moments and the
        # gradients move once a batch; forward and two backward products
        return {"bytes": case["epochs"] * (4.0 * rows * (i + o) + batches * 24.0 * weights),
                "flops": 6.0 * weights * rows * case["epochs"]}
    if kind in ("ensemble", "closure"):
        nodes = sum(math.comb(d + l - 1, l - 1) for l in _depths(case))
    else:
        nodes = math.comb(d + case["lh"] - 1, case["lh"] - 1)
    # A Hermitian ADO holds N^2 real values.
    el = float(nodes) * n * n
    rhs = nodes * (8.0 * n ** 3 + 16.0 * n * d + 16.0 * n * n)
    b = 4.0 if case["precision"] == "fp32" else 8.0
    if kind == "rhs":
        return {"bytes": 32.0 * el, "flops": 2 * rhs}
    if kind == "steady":
        # BiCGSTAB(2): about 100 cycles of four products and eight vector passes
        return {"bytes": 100 * 12 * 16.0 * el, "flops": 100 * 4 * rhs}
    if kind == "rkf45":
        # state in and out; per stage its input and output
        return {"bytes": case["steps"] * el * (16.0 + 6 * 2 * b), "flops": case["steps"] * 6 * rhs}
    step = {"bytes": el * (16.0 + 6 * b), "flops": 4.0 * rhs}
    if kind == "bath":
        step["flops"] += 4.0 * nodes * n * 32.0 * n ** 3
    if kind == "closure":
        i, h, o = _net_sizes(case)
        rows = case["members"] * math.comb(d + case["lh"] - 2, case["lh"] - 1)
        step["flops"] += 4.0 * rows * 2.0 * (i * h + h * h + h * 2 * n * d)
        step["bytes"] += 4.0 * rows * 4.0 * 2 * n * d
    return {k: v * case["steps"] for k, v in step.items()}


def tolerance(case):
    """About four times what the paths show against exact(), or, for the
    training, against the same rows summed in another order."""
    kind = case["kind"]
    if kind == "train":
        # bfloat16 operands: a last-bit change of an FP32 sum flips roundings,
        # and Adam's normalised steps carry it on
        return {"rel": 2e-4, "max": 6e-3}
    if kind == "steady":
        # any state whose residual is below the solver's 1e-10
        return {"rel": 1e-9, "max": 1e-8}
    if kind == "rkf45":
        # the error estimate is a difference of nearly equal values
        return {"rel": 4e-8, "max": 8e-8}
    if case["precision"] == "fp32":
        return {"rel": 1e-6, "max": 4e-6}
    return {"rel": 3e-14, "max": 4e-13}


# --- The same in plain torch, 64 bits ------------------------------------------------

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _enumerate(d, lh):
    """Multi-indices in PHI's order (hierarchy.cc:45-155)."""
    idx = [(0,) * d]
    seen = {idx[0]: 0}
    level = [0]
    for t in range(1, lh):
        new = []
        if t == 1:
            cand = [(0, j) for j in range(d)]
        else:
            cand = [(p, (q + k) % d) for k in range(d) for q, p in enumerate(level)]
        for p, j in cand:
            v = list(idx[p])
            v[j] += 1
            v = tuple(v)
            if v not in seen:
                seen[v] = len(idx)
                new.append(len(idx))
                idx.append(v)
        level = new
    return idx, seen


class _Heom:
    """PHI's independent-bath (or full-operator) equations on states of shape
    (members, nodes, N, N); a call gives their right-hand side."""

    def __init__(self, case, Hs, lh, ops=None):
        n, K = case["sites"], case["terms"]
        d = n * K
        dev = self.dev = _device()
        idx, seen = _enumerate(d, lh)
        self.idx = np.array(idx)
        self.n, self.K, self.d, self.nodes = n, K, d, len(idx)
        thermal = KB * case["temp"]
        nu = 2 * math.pi * thermal / HBAR
        lam, g = case["lam"], case["gam"]
        corr = np.zeros(K, dtype=complex)
        corr[0] = g * lam / HBAR * complex(1 / math.tan(g * HBAR / (2 * thermal)), -1)
        delta = 2 * lam * thermal / HBAR ** 2 / g - lam / HBAR / math.tan(HBAR * g / (2 * thermal))
        for k in range(1, K):
            corr[k] = 4 * lam * g * thermal / HBAR ** 2 * nu * k / ((nu * k) ** 2 - g ** 2)
            delta -= 4 * lam * thermal / HBAR ** 2 * g / ((nu * k) ** 2 - g ** 2)
        self.delta, vacuum = delta, lh == 1
        rate = np.array([g if k == 0 else nu * k for k in range(K)] * n)
        self.mu = torch.tensor(self.idx @ rate, device=dev)[None, :, None, None]
        none = len(idx)
        tier = self.idx.sum(axis=1)
        nxt = np.full((d, none), none)
        prv = np.full((d, none), none)
        sn, sc, sr = (np.zeros((d, none)), np.zeros((d, none), complex), np.zeros((d, none), complex))
        for i, v in enumerate(idx):
            for j in range(d):
                c = corr[j % K]
                if v[j] > 0:
                    prv[j, i] = seen[v[:j] + (v[j] - 1,) + v[j + 1:]]
                    q = v[j] / math.sqrt(v[j] * abs(c))
                    sr[j, i] = 1j * c * q
                    sc[j, i] = -1j * np.conj(c) * q
                if tier[i] < lh - 1:
                    nxt[j, i] = seen[v[:j] + (v[j] + 1,) + v[j + 1:]]
                sn[j, i] = math.sqrt((v[j] + 1) * abs(c))
        t = lambda a: torch.tensor(a, device=dev)  # noqa: E731
        self.nxt, self.prv, self.sn, self.sc, self.sr = t(nxt), t(prv), t(sn), t(sc), t(sr)
        self.H = torch.tensor(np.asarray(Hs), dtype=torch.complex128, device=dev)[:, None]
        off = np.ones((n, n)) - np.eye(n)
        self.deph = t(2 * delta * off)[None, None]
        self.ops = None if ops is None else torch.tensor(ops, dtype=torch.complex128, device=dev)

    def left(self, A, x):
        return torch.matmul(A, x)

    def __call__(self, x):
        H, n = self.H, self.n
        k = torch.matmul(H, x) - torch.matmul(x, H)
        k = (-1j / HBAR) * k - self.mu * x
        zero = torch.zeros_like(x[:, :1])
        xp = torch.cat([x, zero], dim=1)
        if self.ops is not None:
            for j in range(self.d):
                F = self.ops[j // self.K]
                u = xp[:, self.nxt[j]] * self.sn[j][None, :, None, None]
                w = xp[:, self.prv[j]]
                k += -1j * (torch.matmul(F, u) - torch.matmul(u, F))
                k -= (self.sr[j][None, :, None, None] * torch.matmul(F, w)
                      + self.sc[j][None, :, None, None] * torch.matmul(w, F))
            for F in self.ops:
                c = torch.matmul(F, x) - torch.matmul(x, F)
                k -= self.delta * (torch.matmul(F, c) - torch.matmul(c, F))
            return k
        k = k - self.deph * x
        for j in range(self.d):
            b = j // self.K
            s, c, r = (v[j][None, :, None] for v in (self.sn, self.sc, self.sr))
            col, row = xp[:, :, :, b], xp[:, :, b, :]
            k[:, :, :, b] += 1j * s * col[:, self.nxt[j]] - c * col[:, self.prv[j]]
            k[:, :, b, :] -= 1j * s * row[:, self.nxt[j]] + r * row[:, self.prv[j]]
        return k

    def start(self):
        x = torch.zeros((self.H.shape[0], self.nodes, self.n, self.n), dtype=torch.complex128,
                        device=self.dev)
        x[:, 0, 0, 0] = 1.0
        return x


def _rk4(f, x, dt):
    k0 = f(x)
    k1 = f(x + dt / 2 * k0)
    k2 = f(x + dt / 2 * k1)
    k3 = f(x + dt * k2)
    return x + dt / 6 * (k0 + 2 * k1 + 2 * k2 + k3)


class _Closed(_Heom):
    """The hierarchy whose last tier reads the network's predictions."""

    def __init__(self, case, Hs, lh, flat):
        super().__init__(case, Hs, lh)
        i, h, o = _net_sizes(case)
        f, w = np.asarray(flat, dtype=np.float64), []
        for shape in ((h, i), (h,), (h, h), (h,), (o, h), (o,)):
            m = int(np.prod(shape))
            w.append(torch.tensor(f[:m].reshape(shape), device=self.dev))
            f = f[m:]
        self.w = w
        last = np.nonzero(self.idx.sum(axis=1) == lh - 1)[0]
        self.first = int(last[0])
        self.occ = torch.tensor(self.idx[last] / (lh - 1.0), device=self.dev)
        self.sb = self.sn[:, self.first:]

    def __call__(self, x):
        k = super().__call__(x)
        m, n, d = x.shape[0], self.n, self.d
        b = x[:, self.first:]
        s = torch.maximum(b.real.abs(), b.imag.abs()).amax(dim=(2, 3)).clamp_min(1e-30)
        v = (b / s[:, :, None, None]).transpose(2, 3).reshape(m, -1, n * n)
        z = torch.cat([v.real, v.imag, self.occ.expand(m, -1, -1)], dim=2)
        w = self.w
        z = torch.nn.functional.gelu(z @ w[0].T + w[1])
        z = torch.nn.functional.gelu(z @ w[2].T + w[3])
        z = (z @ w[4].T + w[5]).reshape(m, -1, d, 2, n, n)  # mode, re/im, column, row
        y = torch.complex(z[:, :, :, 0], z[:, :, :, 1]) * s[:, :, None, None, None]
        for j in range(d):
            c = j // self.K
            t = 1j * self.sb[j][None, :, None] * y[:, :, j, c, :]
            k[:, self.first:, :, c] += t
            k[:, self.first:, c, :] += t.conj()
        return k


def _history(f, x, case, dt):
    hist = []
    for i in range(case["steps"]):
        x = _rk4(f, x, dt)
        if i % case["every"] == 0:
            hist.append(x[:, 0].clone())
    return torch.stack(hist, dim=1), x


def exact(case, seed):
    kind, dt = case["kind"], 0.001
    if kind == "train":
        return None  # the library's own shuffle decides the minibatches
    if kind in ("ensemble", "closure"):
        Hs, depths = _members(case, seed), np.array(_depths(case))
        hist, last = None, np.zeros((len(Hs),) + Hs[0].shape, dtype=complex)
        for lh in sorted(set(depths)):
            who = np.nonzero(depths == lh)[0]
            for part in np.array_split(who, max(1, len(who) // 64)):
                if kind == "closure":
                    f = _Closed(case, Hs[part], int(lh), _net_params(case, seed))
                else:
                    f = _Heom(case, Hs[part], int(lh))
                h, x = _history(f, f.start(), case, dt)
                h = h.sum(dim=0)
                hist = h if hist is None else hist + h
                last[part] = x[:, 0].cpu().numpy()
        return [(hist / len(Hs)).cpu().numpy(), last]
    rng = _rng(case, seed)
    H = _hamiltonian(case, rng)
    f = _Heom(case, [H], case["lh"], _bath_ops(case, rng) if kind == "bath" else None)
    if kind == "rhs":
        x = torch.tensor(_rhs_input(case, seed), device=f.dev)[None]
        return [f(x)[0].cpu().numpy()]
    x = f.start()
    if kind in ("rk4", "bath"):
        h, x = _history(f, x, case, dt)
        return [h[0].cpu().numpy(), (x[0] if case["state"] else x[0, 0]).cpu().numpy()]
    if kind == "launch":
        for _ in range(case["steps"]):
            x = _rk4(f, x, dt)
        return [x[0, 0].cpu().numpy(), x[0].cpu().numpy()]
    if kind == "rkf45":
        c = _rkf45_coefs(dt)
        b = [c[s * (s + 1) // 2:(s + 1) * (s + 2) // 2] for s in range(5)]
        c4, c5, errs = c[15:19], c[19:], []
        for _ in range(case["steps"]):
            k = [f(x)]
            for s in range(5):
                k.append(f(x + sum(w * q for w, q in zip(b[s], k))))
            y4 = x + sum(w * k[i] for w, i in zip(c4, (0, 2, 3, 4)))
            y5 = x + sum(w * k[i] for w, i in zip(c5, (0, 2, 3, 4, 5)))
            errs.append(float((y4 - y5).abs().max()))
            x = y5
        return [np.array(errs), x[0, 0].cpu().numpy()]
    # steady: long BiCGSTAB in 64 bits to a residual far below the solver's
    # (the element (0, 0) of node 0 replaced by the trace)
    def op(v):
        y = f(v)
        y[0, 0, 0, 0] = torch.diagonal(v[0, 0]).sum()
        return y

    def dot(a, c):
        return torch.vdot(a.reshape(-1), c.reshape(-1))

    rhs = torch.zeros_like(x)
    rhs[0, 0, 0, 0] = 1.0
    r = rhs - op(x)
    best, rh, p = (float(r.norm()), x), r.clone(), r.clone()
    rho = dot(rh, r)
    for _ in range(600):
        v = op(p)
        a = rho / dot(rh, v)
        s = r - a * v
        t = op(s)
        w = dot(t, s) / dot(t, t)
        x = x + a * p + w * s
        r = s - w * t
        new = dot(rh, r)
        p = r + (new / rho) * (a / w) * (p - w * v)
        rho = new
        if float(r.norm()) < best[0]:
            best = (float(r.norm()), x)
        if best[0] < 1e-12:
            break
    return [None, best[1][0, 0].cpu().numpy()] if best[0] < 1e-11 else None
