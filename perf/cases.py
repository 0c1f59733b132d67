"""The framework's work, case by case, for timing it and comparing its results.

A case is a dict of plain values; ``prepare`` makes what a program has in hand
before the call, ``run`` is the call.  The kinds, and what each stands for:

  orbit              Hamiltonian.integrate_orbit with Leapfrog, the trajectory
                     as host arrays: one orbit at the prompt, small ensembles
  orbit_dop853       the same with DOP853 (gala's batches of 100 orbits by
                     default, every orbit on its own with nbatch=1)
  field              PotentialBase.energy and .gradient at host positions: maps
                     of a potential, labels for a fit
  leapfrog           integrate.leapfrog on device states, final states or a
                     saved trajectory, in the composite or an SCF expansion
  dop853             integrate.dop853 over orbits of uneven length
  dop853_batched     integrate.dop853_batched, the default batching at scale
  mockstream         MockStreamGenerator.run, progenitor to final stream
  surrogate_train    one training step: gradients and Adam
  surrogate_forward  the network's potential and its gradient
  surrogate_leapfrog orbits on the network with the exact-force fallback

Sizes follow the benchmark workloads (gala_amd/workloads.py), the tests and
the README example, and the range around them.
"""
import math

import numpy as np
import torch

from gala_amd import workloads
from gala_amd.dynamics import FardalStreamDF, MockStreamGenerator
from gala_amd.integrate import dop853, dop853_batched, leapfrog
from gala_amd.potential import (Hamiltonian, HernquistPotential, MilkyWayLikePotential,
                                MiyamotoNagaiPotential, NFWPotential, PlummerPotential,
                                SCFPotential)
from gala_amd.surrogate import PARAM_SHAPES, SCFSurrogate, init_params
from gala_amd.units import G

SCF_M, SCF_RS = 1e12, 20.0
SINGLE = {"hernquist": {"m": 1e12, "c": 20.0}, "plummer": {"m": 1e11, "b": 5.0},
          "miyamotonagai": {"m": 6.8e10, "a": 3.0, "b": 0.28}, "nfw": {"m": 5.4e11, "r_s": 15.6}}


def listed():
    return [
        # one orbit in the composite, 1 Gyr: the README's call, all latency
        {"name": "orbit_one", "kind": "orbit", "pot": "composite", "n": 1, "n_steps": 1000,
         "dt": 1.0},
        # a handful of orbits with the adaptive integrator and its default
        # batches, a ragged last one, dense output at every time
        {"name": "orbits_dop853", "kind": "orbit_dop853", "n": 137, "n_steps": 500, "dt": 1.0,
         "nbatch": 100},
        # energies and forces of a moderate expansion at scattered positions
        {"name": "scf_field", "kind": "field", "pot": "scf", "n": 100001, "nmax": 6, "lmax": 4},
        # the 1,024-orbit Leapfrog workload, every step kept on the device
        {"name": "leapfrog_saved", "kind": "leapfrog", "pot": "composite", "n": 1024,
         "n_steps": 10000, "dt": 1.0, "stride": 1},
        # a large ensemble, final states only
        {"name": "leapfrog_final", "kind": "leapfrog", "pot": "composite", "n": 1048576,
         "n_steps": 1000, "dt": 1.0, "stride": 0},
        # the SCF Leapfrog workload over its first 100 Myr
        {"name": "scf_leapfrog", "kind": "leapfrog", "pot": "scf", "n": 262144, "n_steps": 200,
         "dt": 0.5, "stride": 0, "nmax": 10, "lmax": 6},
        # the uneven DOP853 workload, longest first by a pilot pass
        {"name": "dop853_uneven", "kind": "dop853", "n": 1048576},
        # gala's default batching at scale
        {"name": "dop853_batched", "kind": "dop853_batched", "n": 262144, "t1": 1000.0,
         "nbatch": 100},
        # the mock-stream workload, end to end
        {"name": "mockstream", "kind": "mockstream", "integrator": "leapfrog", "n_steps": 4000},
        # one step of the surrogate's training loop at its batch size
        {"name": "surrogate_train", "kind": "surrogate_train", "m": 32768},
        # a large inference batch
        {"name": "surrogate_forward", "kind": "surrogate_forward", "m": 1048576},
        # orbits on the network, some of which fall back
        {"name": "surrogate_leapfrog", "kind": "surrogate_leapfrog", "n": 65537, "n_steps": 50,
         "dt": 0.5, "tol": 1e-5},
    ]


def _log_int(rng, lo, hi):
    """a whole number spread over [lo, hi] by its logarithm, odd as often as even"""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["orbit", "orbit_dop853", "field", "leapfrog", "leapfrog", "scf", "scf",
                       "dop853", "dop853_batched", "mockstream", "surrogate_train",
                       "surrogate_forward", "surrogate_leapfrog"])
    if kind == "orbit":
        n = _log_int(rng, 1, 512)
        return {"kind": kind, "pot": rng.choice(["composite"] + sorted(SINGLE)), "n": n,
                "n_steps": _log_int(rng, 50, 4000), "dt": rng.choice([0.5, 1.0, -1.0])}
    if kind == "orbit_dop853":
        return {"kind": kind, "n": _log_int(rng, 1, 1000), "n_steps": _log_int(rng, 20, 1000),
                "dt": 1.0, "nbatch": rng.choice([100, 100, 1])}
    if kind == "field":
        case = {"kind": kind, "pot": rng.choice(["composite", "scf", "scf"] + sorted(SINGLE)),
                "n": _log_int(rng, 1, 1000000)}
        if case["pot"] == "scf":
            case.update(nmax=rng.randint(2, 14), lmax=rng.randint(0, 8))
        return case
    if kind == "leapfrog":
        n = _log_int(rng, 64, 1048576)
        steps = min(10000, _log_int(rng, 100, 10000), max(100, int(1.0e9 / n)))
        stride = rng.choice([0, 0, 1, 4, 16])
        if stride and 48.0 * n * steps / stride > 2e9:
            stride = 0
        return {"kind": kind, "pot": rng.choice(["composite", "composite"] + sorted(SINGLE)),
                "n": n, "n_steps": steps, "dt": 1.0, "stride": stride}
    if kind == "scf":
        nmax, lmax = rng.choice([(10, 6), (rng.randint(2, 14), rng.randint(0, 8))])
        n = _log_int(rng, 64, 262144)
        terms = (nmax + 1) * (lmax + 1) * (lmax + 2) / 2
        steps = max(4, min(1000, int(100 * 262144 / n * min(1.0, 308.0 / terms))))
        return {"kind": "leapfrog", "pot": "scf", "n": n, "n_steps": steps, "dt": 0.5,
                "stride": rng.choice([0, 0, 4]), "nmax": nmax, "lmax": lmax}
    if kind == "dop853":
        return {"kind": kind, "n": _log_int(rng, 1000, 1048576)}
    if kind == "dop853_batched":
        return {"kind": kind, "n": _log_int(rng, 1000, 262144),
                "t1": float(rng.choice([100.0, 300.0, 1000.0])),
                "nbatch": rng.choice([16, 37, 64, 100, 100, 300])}
    if kind == "mockstream":
        return {"kind": kind, "integrator": rng.choice(["leapfrog", "leapfrog", "dop853"]),
                "n_steps": _log_int(rng, 200, 4000)}
    if kind == "surrogate_train":
        return {"kind": kind, "m": 64 * _log_int(rng, 16, 1024)}
    if kind == "surrogate_forward":
        return {"kind": kind, "m": _log_int(rng, 1, 1048576)}
    return {"kind": kind, "n": _log_int(rng, 1000, 262144), "n_steps": rng.randint(5, 40),
            "dt": 0.5, "tol": rng.choice([1e-5, 1e-4, 1e300])}


# ---------------------------------------------------------------------------
# inputs

def _vcirc(name):
    """circular speed at (3, n) positions, from the closed forms (the SCF
    expansion's monopole stands for the expansion)"""
    if name == "scf":
        grad = _component_grad("hernquist", {"m": SCF_M, "c": SCF_RS})
        grads = [grad]
    elif name == "composite":
        grads = [_component_grad(k, p) for k, p in workloads.MW_COMPONENTS]
    else:
        grads = [_component_grad(name, SINGLE[name])]

    def fn(q):
        x, y, z = (torch.from_numpy(np.ascontiguousarray(c)) for c in q)
        r = torch.sqrt(x * x + y * y + z * z)
        g = sum(a * x + b * y + c * z for a, b, c in (f(x, y, z) for f in grads))
        return torch.sqrt(g.abs()).numpy() if len(r) else np.zeros(0)
    return fn


def _states(case, seed):
    """(6, n) initial states: the workloads' radii and speeds"""
    rng = np.random.default_rng(seed)
    n, name = case["n"], case.get("pot", "composite")
    if name == "scf":
        r = np.exp(rng.uniform(np.log(2.0), np.log(150.0), n))
    else:
        r = rng.uniform(5.0, 30.0, n)
    return workloads.initial_conditions(rng, n, r, _vcirc(name), 0.1)


def _potential(case, seed):
    name = case.get("pot", "composite")
    if name == "composite":
        return MilkyWayLikePotential()
    if name == "scf":
        S, T = workloads.scf_coefficients(case.get("nmax", 10), case.get("lmax", 6), seed)
        return SCFPotential(m=SCF_M, r_s=SCF_RS, Snlm=S, Tnlm=T)
    cls = {"hernquist": HernquistPotential, "plummer": PlummerPotential,
           "miyamotonagai": MiyamotoNagaiPotential, "nfw": NFWPotential}[name]
    return cls(**SINGLE[name])


def _positions(rng, n, lo, hi):
    r = np.exp(rng.uniform(math.log(lo), math.log(hi), n))
    u = rng.normal(size=(3, n))
    return np.ascontiguousarray(u / np.linalg.norm(u, axis=0) * r)


def _network(seed):
    """parameters of a network in use: the initial distribution with an output
    layer that has grown to outputs of order one"""
    theta = init_params(seed)
    theta[-(256 * 4 + 4):-4] *= 10.0
    return theta


def _adam_state(seed):
    """first and second moments as a run has them after some steps"""
    rng = np.random.default_rng(seed + 7)
    n = sum(int(np.prod(s)) for _, s in PARAM_SHAPES)
    m = (1e-3 * rng.normal(size=n)).astype(np.float32)
    v = (1e-5 * rng.uniform(0.5, 2.0, n)).astype(np.float32)
    return m, v


def _train_batch(case, seed):
    """features and targets of a batch: unit directions and standardised log
    radii; a smooth field of them plus scatter"""
    rng = np.random.default_rng(seed)
    u = rng.normal(size=(case["m"], 3))
    u /= np.linalg.norm(u, axis=1)[:, None]
    f = np.concatenate([u, rng.uniform(-1.7, 1.7, (case["m"], 1))], axis=1)
    k = rng.normal(size=(4, 4))
    t = np.sin(f @ k) + 0.1 * rng.normal(size=(case["m"], 4))
    return f.astype(np.float32), t.astype(np.float32)


ADAM_STEP, ADAM_LR = 100, 1e-3


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    if kind in ("orbit", "orbit_dop853"):
        state["H"] = Hamiltonian(_potential(case, seed))
        state["w0"] = _states(case, seed)
    elif kind == "field":
        state["pot"] = _potential(case, seed)
        state["q"] = _positions(np.random.default_rng(seed + 1), case["n"], 1.0, 200.0)
    elif kind == "leapfrog":
        state["pot"] = _potential(case, seed)
        state["w0"] = torch.from_numpy(_states(case, seed)).cuda()
    elif kind == "dop853":
        state["pot"] = MilkyWayLikePotential()
        w0, T = workloads.composite_dop853(_vcirc("composite"), n=case["n"], seed=seed)
        state["w0"] = torch.from_numpy(w0).cuda()
        state["t0"] = torch.zeros(case["n"], dtype=torch.float64, device="cuda")
        state["t1"] = torch.from_numpy(T).cuda()
    elif kind == "dop853_batched":
        state["pot"] = MilkyWayLikePotential()
        w0, _ = workloads.composite_dop853(_vcirc("composite"), n=case["n"], seed=seed)
        state["w0"] = torch.from_numpy(w0).cuda()
    elif kind == "mockstream":
        state["H"] = Hamiltonian(MilkyWayLikePotential())
        w0, state["mass"], b, _, _ = workloads.mockstream_progenitor()
        rng = np.random.default_rng(seed)
        state["w0"] = w0 * (1.0 + 0.05 * rng.uniform(-1.0, 1.0, 6))
        state["prog"] = PlummerPotential(m=state["mass"], b=b)
        state["seed"] = seed % (1 << 31)
    elif kind.startswith("surrogate"):
        sur = SCFSurrogate(_potential({"pot": "scf"}, seed))
        sur.set_params(_network(seed))
        state["sur"] = sur
        if kind == "surrogate_train":
            f, t = _train_batch(case, seed)
            state["feat"], state["target"] = torch.from_numpy(f).cuda(), torch.from_numpy(t).cuda()
            m, v = _adam_state(seed)
            sur.m.copy_(torch.from_numpy(m))
            sur.v.copy_(torch.from_numpy(v))
            sur.step = ADAM_STEP
        elif kind == "surrogate_forward":
            q = _positions(np.random.default_rng(seed + 1), case["m"], 1.0, 200.0)
            state["q"] = torch.from_numpy(q).cuda()
        else:
            w0 = _states(dict(case, pot="scf"), seed)
            state["w0"] = torch.from_numpy(w0).cuda()
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "orbit":
        o = state["H"].integrate_orbit(state["w0"], Integrator="leapfrog", dt=case["dt"],
                                       n_steps=case["n_steps"])
        return o.t, o.xyz, o.v_xyz
    if kind == "orbit_dop853":
        kw = {} if case["nbatch"] == 100 else {"nbatch": case["nbatch"]}
        o = state["H"].integrate_orbit(state["w0"], Integrator="dopri853", Integrator_kwargs=kw,
                                       dt=case["dt"], n_steps=case["n_steps"])
        return o.t, o.xyz, o.v_xyz
    if kind == "field":
        return state["pot"].energy(state["q"]), state["pot"].gradient(state["q"])
    if kind == "leapfrog":
        stride = case["stride"]
        return leapfrog(state["pot"], state["w0"], case["dt"], case["n_steps"],
                        save_stride=max(stride, 1), save=stride > 0)
    if kind == "dop853":
        n = case["n"]
        big = n >= 4096  # as integrate_orbit does for many orbits
        r = dop853(state["pot"], state["w0"], state["t0"], state["t1"], 1.0, rtol=1e-8,
                   atol=1e-10, order="pilot" if big else None,
                   n_tail=min(1024, n // 64) if big else 0)
        return r["w_final"], r["status"], r["stats"]
    if kind == "dop853_batched":
        r = dop853_batched(state["pot"], state["w0"], 0.0, case["t1"], 1.0,
                           nbatch=case["nbatch"])
        return r["w_final"], r["status"], r["stats"]
    if kind == "mockstream":
        df = FardalStreamDF(random_state=np.random.RandomState(state["seed"]))
        gen = MockStreamGenerator(df, state["H"], progenitor_potential=state["prog"])
        s, b = gen.run(state["w0"], state["mass"], Integrator=case["integrator"], dt=-1.0,
                       n_steps=case["n_steps"])
        return s.xyz, s.v_xyz, s.release_time, b.xyz, b.v_xyz
    sur = state["sur"]
    if kind == "surrogate_train":
        loss, grad = sur.gradients(state["feat"], state["target"])
        sur.adam(ADAM_LR)
        return loss, grad, sur.theta, sur.m, sur.v
    if kind == "surrogate_forward":
        return sur.forward(state["q"])
    r = sur.leapfrog(state["w0"], case["dt"], case["n_steps"], tol=case["tol"])
    return r["w_final"], r["fallback_step"]


# ---------------------------------------------------------------------------
# work one pass cannot do without (add, multiply, divide, root, log: 1 each,
# fused multiply-add: 2)

GRAD_FLOPS = {"composite": 74, "hernquist": 16, "plummer": 15, "miyamotonagai": 20, "nfw": 22}
NET_PARAMS = sum(int(np.prod(s)) for _, s in PARAM_SHAPES)
NET_MACS = 4 * 256 + 3 * 256 * 256 + 256 * 4


def _grad_flops(case):
    if case.get("pot") != "scf":
        return GRAD_FLOPS[case.get("pot", "composite")]
    nmax, lmax = case["nmax"], case["lmax"]
    L = (lmax + 1) * (lmax + 2) // 2
    return 8 * (nmax + 1) * L + 20 * L + 12 * (nmax + 1) * (lmax + 1) + 8 * L + 50


# accepted DOP853 steps per Myr and orbit over these workloads, per orbit on
# its own at rtol 1e-8 and in batches of 100 at 1e-10 (the finest sets the step)
ACCEPTED_ALONE, ACCEPTED_BATCH = 0.21, 1.48


def work(case):
    kind = case["kind"]
    n, steps = case.get("n", 0), case.get("n_steps", 0)
    if kind == "orbit":
        return {"bytes": 48 * n * (steps + 2), "flops": n * steps * (_grad_flops(case) + 18)}
    if kind == "orbit_dop853":
        per = ACCEPTED_BATCH if case["nbatch"] > 1 else 2 * ACCEPTED_ALONE
        return {"bytes": 48 * n * (steps + 2),
                "flops": int(n * steps * case["dt"] * per * (1840 + 1140))}
    if kind == "field":
        return {"bytes": 8 * n * (3 + 1 + 3), "flops": int(1.5 * n * _grad_flops(case))}
    if kind == "leapfrog":
        saved = steps // case["stride"] + 1 if case["stride"] else 0
        return {"bytes": 48 * n * (2 + saved), "flops": n * steps * (_grad_flops(case) + 18)}
    if kind == "dop853":
        # lengths are log-uniform over 100 to 10,000 Myr: 2,150 on average
        return {"bytes": n * (48 + 24 + 48 + 36),
                "flops": int(n * 2150.0 * ACCEPTED_ALONE * 1840)}
    if kind == "dop853_batched":
        return {"bytes": n * (48 + 48 + 36), "flops": int(n * case["t1"] * ACCEPTED_BATCH * 1840)}
    if kind == "mockstream":
        p = 2 * (steps + 1)  # particles, each over half the span on average
        per = 110 if case["integrator"] == "leapfrog" else 600
        return {"bytes": 2 * 48 * p + 48 * (steps + 1), "flops": p * steps // 2 * per}
    if kind == "surrogate_train":
        m = case["m"]
        return {"bytes": 32 * m + 4 * 8 * NET_PARAMS, "flops": 6 * m * NET_MACS}
    if kind == "surrogate_forward":
        m = case["m"]
        return {"bytes": 8 * m * (3 + 1 + 3) + 4 * NET_PARAMS, "flops": 4 * m * NET_MACS}
    return {"bytes": 48 * 2 * n + 4 * n, "flops": 4 * n * steps * NET_MACS}


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch

def _component_grad(name, p):
    gm = G * p["m"]

    def spherical(f):
        def grad(x, y, z):
            fac = f(torch.sqrt(x * x + y * y + z * z))
            return fac * x, fac * y, fac * z
        return grad

    if name == "hernquist":
        return spherical(lambda r: gm / (r * (r + p["c"]) ** 2))
    if name == "plummer":
        return spherical(lambda r: gm / ((r * r + p["b"] ** 2) * torch.sqrt(r * r + p["b"] ** 2)))
    if name == "nfw":
        def nfw(r):
            u = r / p["r_s"]
            return gm / r ** 3 * (torch.log(1.0 + u) - u / (1.0 + u))
        return spherical(nfw)

    def disk(x, y, z):
        s = torch.sqrt(z * z + p["b"] ** 2)
        d = x * x + y * y + (p["a"] + s) ** 2
        fac = gm / (d * torch.sqrt(d))
        return fac * x, fac * y, fac * z * (1.0 + p["a"] / s)
    return disk


def _component_value(name, p, x, y, z):
    gm = G * p["m"]
    r = torch.sqrt(x * x + y * y + z * z)
    if name == "hernquist":
        return -gm / (r + p["c"])
    if name == "plummer":
        return -gm / torch.sqrt(r * r + p["b"] ** 2)
    if name == "nfw":
        return -gm / r * torch.log(1.0 + r / p["r_s"])
    s = p["a"] + torch.sqrt(z * z + p["b"] ** 2)
    return -gm / torch.sqrt(x * x + y * y + s * s)


def _scf_field(S, T, want_value=True):
    """(x, y, z) -> value, (gx, gy, gz) of the Hernquist-Ostriker expansion:
    Phi = (G M / r_s) sum_lm Y_lm (A_lm cos m phi + B_lm sin m phi) with
    A_lm = sum_n phi_nl S_nlm, phi_nl = -sqrt(4 pi) s^l (1 + s)^(-2l-1)
    C_n^(2l+3/2)(xi), xi = (s - 1) / (s + 1)."""
    nmax, lmax = S.shape[0] - 1, S.shape[1] - 1
    gm = G * SCF_M
    # per l, the (2 (l + 1), nmax + 1) matrix of S and T over n
    coef = [torch.from_numpy(np.ascontiguousarray(
        np.concatenate([S[:, l, :l + 1], T[:, l, :l + 1]], axis=1).T)).cuda()
        for l in range(lmax + 1)]

    def gegenbauer(a, xi, count):
        rows = [torch.ones_like(xi)]
        if count > 1:
            rows.append(2.0 * a * xi)
        for n in range(2, count):
            rows.append((2.0 * (n + a - 1.0) * xi * rows[-1] - (n + 2.0 * a - 2.0) * rows[-2]) / n)
        return torch.stack(rows[:count]) if count > 0 else None

    def field(x, y, z):
        R2 = x * x + y * y
        r, R = torch.sqrt(R2 + z * z), torch.sqrt(R2)
        s, ct, st = r / SCF_RS, z / r, R / r
        cp, sp = x / R, y / R
        one = 1.0 + s
        xi = (s - 1.0) / one
        cm, sm = [torch.ones_like(x)], [torch.zeros_like(x)]
        for m in range(1, lmax + 1):
            cm.append(cm[-1] * cp - sm[-1] * sp)
            sm.append(sm[-1] * cp + cm[-2] * sp)
        phi, dr = torch.zeros_like(x), torch.zeros_like(x)
        dth, dph = torch.zeros_like(x), torch.zeros_like(x)
        prev = []
        prev2 = []
        diag = torch.full_like(x, 1.0 / math.sqrt(4.0 * math.pi))
        for l in range(lmax + 1):
            a = 2.0 * l + 1.5
            pre = -math.sqrt(4.0 * math.pi) * s ** l / one ** (2 * l + 1)
            C = gegenbauer(a, xi, nmax + 1)
            A = pre * (coef[l] @ C)
            dA = (l / s - (2 * l + 1.0) / one) * A
            if nmax > 0:
                dA = dA + pre * (4.0 * a / one ** 2) * (
                    coef[l][:, 1:].contiguous() @ gegenbauer(a + 1.0, xi, nmax))
            Y = []
            for m in range(l + 1):
                if m == l:
                    Y.append(diag)
                elif m == l - 1:
                    Y.append(math.sqrt(2.0 * m + 3.0) * ct * prev[m])
                else:
                    k = math.sqrt((4.0 * l * l - 1.0) / (l * l - m * m))
                    b = math.sqrt(((l - 1.0) ** 2 - m * m) / (4.0 * (l - 1.0) ** 2 - 1.0))
                    Y.append(k * (ct * prev[m] - b * prev2[m]))
            for m in range(l + 1):
                Am, Bm = A[m], A[l + 1 + m]
                both = Am * cm[m] + Bm * sm[m]
                phi = phi + Y[m] * both
                dr = dr + Y[m] * (dA[m] * cm[m] + dA[l + 1 + m] * sm[m])
                dY = l * ct * Y[m]  # sin(theta) dY/dtheta
                if m < l:
                    dY = dY - math.sqrt((2.0 * l + 1.0) / (2.0 * l - 1.0) * (l * l - m * m)) * prev[m]
                dth = dth + dY * both
                dph = dph + m * Y[m] * (Bm * cm[m] - Am * sm[m])
            prev2, prev = prev, Y
            diag = -math.sqrt((2.0 * l + 3.0) / (2.0 * l + 2.0)) * st * diag
        gr, gt, gp = dr, dth / (s * st), dph / (s * st)
        fac = gm / SCF_RS ** 2
        return (phi * (gm / SCF_RS),
                ((st * cp * gr + ct * cp * gt - sp * gp) * fac,
                 (st * sp * gr + ct * sp * gt + cp * gp) * fac,
                 (ct * gr - st * gt) * fac))
    return field


def _field(case, seed):
    """(x, y, z) -> value, gradient of the case's potential"""
    name = case.get("pot", "composite")
    if name == "scf":
        return _scf_field(*workloads.scf_coefficients(case.get("nmax", 10), case.get("lmax", 6),
                                                      seed))
    parts = workloads.MW_COMPONENTS if name == "composite" else ((name, SINGLE[name]),)
    grads = [_component_grad(k, p) for k, p in parts]

    def field(x, y, z):
        gs = [g(x, y, z) for g in grads]
        return (sum(_component_value(k, p, x, y, z) for k, p in parts),
                tuple(sum(g[c] for g in gs) for c in range(3)))
    return field


def _leapfrog_exact(field, w0, dt, n_steps, stride):
    """saved rows (6, n_steps // stride + 1, n) (None for stride 0), final (6, n)"""
    x, v = list(w0[:3]), list(w0[3:])
    rows = None
    if stride:
        rows = torch.empty((6, n_steps // stride + 1, w0.shape[1]), dtype=w0.dtype,
                           device=w0.device)
        rows[:, 0] = w0
    g = field(*x)[1]
    h = [v[c] - g[c] * (0.5 * dt) for c in range(3)]
    for j in range(1, n_steps + 1):
        x = [x[c] + h[c] * dt for c in range(3)]
        g = field(*x)[1]
        v = [h[c] - g[c] * (0.5 * dt) for c in range(3)]
        h = [h[c] - g[c] * dt for c in range(3)]
        if stride and j % stride == 0:
            rows[:, j // stride] = torch.stack(x + v)
    return rows, torch.stack(x + v)


def _unpack64(theta):
    out, o = {}, 0
    for name, shape in PARAM_SHAPES:
        k = int(np.prod(shape))
        out[name] = torch.from_numpy(theta[o:o + k].reshape(shape)).cuda().double()
        o += k
    return out


def _layers(p, f):
    h = f
    for l in range(1, 5):
        h = torch.nn.functional.silu(h @ p[f"W{l}"] + p[f"b{l}"])
    return h @ p["W5"] + p["b5"]


def _train_exact(case, seed):
    f, t = (torch.from_numpy(a).cuda().double() for a in _train_batch(case, seed))
    p = _unpack64(_network(seed))
    for a in p.values():
        a.requires_grad_(True)
    loss = ((_layers(p, f) - t) ** 2).sum()
    (loss / case["m"]).backward()
    g = torch.cat([p[name].grad.reshape(-1) for name, _ in PARAM_SHAPES])
    m, v = (torch.from_numpy(a).cuda().double() for a in _adam_state(seed))
    m = 0.9 * m + 0.1 * g
    v = 0.999 * v + 0.001 * g * g
    k = ADAM_STEP + 1
    theta = torch.from_numpy(_network(seed)).cuda().double()
    theta = theta - ADAM_LR * (m / (1.0 - 0.9 ** k)) / (torch.sqrt(v / (1.0 - 0.999 ** k)) + 1e-8)
    return loss.detach().reshape(1), g, theta, m, v


def _forward_exact(case, seed):
    scf = {"pot": "scf"}
    lo, hi = math.log(1.0), math.log(200.0)
    # the network's scale: RMS of Phi / Phi_b - 1 over its radii
    qs = torch.from_numpy(_sample(1 << 16, 20240)).cuda()
    gm = G * SCF_M
    r = torch.sqrt((qs * qs).sum(0))
    c = torch.sqrt(torch.mean((_field(scf, seed)(*qs)[0] / (-gm / (r + SCF_RS)) - 1.0) ** 2))
    p = _unpack64(_network(seed))
    q = torch.from_numpy(_positions(np.random.default_rng(seed + 1), case["m"], 1.0, 200.0)).cuda()
    phi, grad = torch.empty_like(q[0]), torch.empty_like(q)
    for i in range(0, case["m"], 1 << 17):
        x = q[:, i:i + (1 << 17)].clone().requires_grad_(True)
        r = torch.sqrt((x * x).sum(0))
        f = torch.stack([x[0] / r, x[1] / r, x[2] / r,
                         (torch.log(r) - 0.5 * (lo + hi)) * (math.sqrt(12.0) / (hi - lo))], 1)
        v = -gm / (r + SCF_RS) * (1.0 + c * _layers(p, f)[:, 0])
        v.sum().backward()
        phi[i:i + (1 << 17)] = v.detach()
        grad[:, i:i + (1 << 17)] = x.grad
    return phi, grad


def _sample(n, seed):
    """the surrogate's own sample of its radii"""
    rng = np.random.default_rng(seed)
    r = np.exp(rng.uniform(math.log(1.0), math.log(200.0), n))
    u = rng.normal(size=(3, n))
    return u / np.linalg.norm(u, axis=0) * r


def exact(case, seed):
    kind = case["kind"]
    if kind == "orbit":
        t = np.arange(case["n_steps"] + 1) * case["dt"]
        w0 = torch.from_numpy(_states(case, seed)).cuda()
        rows, _ = _leapfrog_exact(_field(case, seed), w0, case["dt"], case["n_steps"], 1)
        rows = rows.cpu().numpy()
        if case["n"] == 1:
            rows = rows[..., 0]
        return t, rows[:3], rows[3:]
    if kind == "field":
        q = _positions(np.random.default_rng(seed + 1), case["n"], 1.0, 200.0)
        v, g = _field(case, seed)(*torch.from_numpy(q).cuda())
        return v.cpu().numpy(), torch.stack(g).cpu().numpy()
    if kind == "leapfrog":
        if case.get("pot") == "scf" and case["n_steps"] > 300:
            return None
        w0 = torch.from_numpy(_states(case, seed)).cuda()
        return _leapfrog_exact(_field(case, seed), w0, case["dt"], case["n_steps"],
                               case["stride"])
    if kind == "surrogate_train":
        return _train_exact(case, seed)
    if kind == "surrogate_forward":
        return _forward_exact(case, seed)
    # the adaptive integrators' steps, the stream's release draws and the
    # switch to the exact force have no closed counterpart
    return None
