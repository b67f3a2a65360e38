"""Performance cases of the TCL4 engine: what its users have it do, through
its public entry points, with sizes from the benchmark, the tests and the
workload generators of this repository.

Kinds of case ("kind"):

  l4       build_l4_dev: L4(t) for many times, inputs resident in HBM
  l4_host  build_TCL4_generator_hip_fused_batch: the same from host arrays
  l4_one   build_TCL4_generator_hip_fused: one time of one system
  run      tcl4_propagate: states r(t) of the TCL2 + L4 run
  batch    Batch.run(graph=True): a set of different systems in one pass
  grad1    SpinPairProblem.loss and its gradient (d = 4)
  gradn    TfimChainProblem.losses_many and its gradients (several sets)
  bath     bath_gamma_hip: C(t) and the Gamma table of a bath
  rk4      propagate_rk4_dense over a caller's generator series

A case fixes the sizes and the Hamiltonian where a program keeps one (a scan
over baths, "scan": "bath"); with "scan": "system" each seed is another
Hamiltonian as well.  The libm phase convention is the library's default;
"phases": "cr" is what large d needs (its phase table would not fit).
"""
import math

import numpy as np
import torch

import taco_amd as taco
from taco_amd import adjoint
from taco_amd import tcl4

SX = np.array([[0, 1], [1, 0]], complex)
SZ = np.array([[1, 0], [0, -1]], complex)


def listed():
    return [
        # one generator of a small system: the shortest call there is
        {"name": "l4_one_d2", "kind": "l4_one", "h": "gue", "d": 2, "ops": 1, "nt": 4096, "dt": 0.005, "t": 1500,
         "scan": "system"},
        # a scan over baths of the spin-boson model: 2000 steps of r(t), host arrays in and out
        {"name": "run_spin_boson", "kind": "run", "h": "spin_boson", "d": 2, "ops": 1, "nt": 16384, "dt": 0.005,
         "steps": 2000, "scan": "bath"},
        # the setting of the reference's published timing: d = 2, 10001 times, host arrays in and out
        {"name": "l4_host_d2_published", "kind": "l4_host", "h": "sx", "d": 2, "ops": 1, "nt": 200001,
         "dt": 0.000625, "tmax": 10000, "tstep": 1, "scan": "bath"},
        # three levels, two coupling operators, a ragged grid, every third time
        {"name": "l4_d3_ops2", "kind": "l4", "h": "gue", "d": 3, "ops": 2, "nt": 24007, "dt": 0.005, "tmax": 5001,
         "tstep": 3, "mode": "parity", "phases": "libm", "scan": "bath"},
        # the headline workload: d = 4, grid 200001, every time to 10000
        {"name": "l4_d4_headline", "kind": "l4", "h": "gue", "d": 4, "ops": 1, "nt": 200001, "dt": 0.002,
         "tmax": 10000, "tstep": 1, "mode": "parity", "phases": "libm", "scan": "bath"},
        # the same with the FFT over the window of the kept times only
        {"name": "l4_d4_window", "kind": "l4", "h": "gue", "d": 4, "ops": 1, "nt": 200001, "dt": 0.002,
         "tmax": 10000, "tstep": 1, "mode": "window", "phases": "libm", "scan": "bath"},
        # eight levels (57 buckets, about 5e4 triples): the large-d end of the batch mix
        {"name": "l4_d8", "kind": "l4", "h": "gue", "d": 8, "ops": 1, "nt": 16384, "dt": 0.005, "tmax": 1000,
         "tstep": 4, "mode": "parity", "phases": "cr", "scan": "bath"},
        # many different small systems at once, L4 and 500 steps each, replayed as a graph
        {"name": "batch_mixed", "kind": "batch", "dims": "2 3 4 2 6 4 3 2 4 3", "log2nt": "14 15 16 17 14 15 16 15 14 17",
         "stride": "1 4 2 8 1 2 4 2 8 1", "n_time": 500, "dt": 0.005},
        # one training step of the d = 4 spin pair at new parameters
        {"name": "grad_spin_pair", "kind": "grad1", "nt": 65536, "dt": 0.005, "steps": 4000},
        # one training step of four parameter sets of the 4-spin chain (d = 16)
        {"name": "grad_chain_d16", "kind": "gradn", "spins": 4, "sets": 4, "nt": 4096, "dt": 0.005, "steps": 200},
        # the Gamma table of a bath on the headline grid
        {"name": "bath_13", "kind": "bath", "nt": 200001, "dt": 0.002, "nf": 13},
        # a caller's own generator series: d = 4, 4000 steps
        {"name": "rk4_d16", "kind": "rk4", "D": 16, "steps": 4000, "dt": 0.005, "every": 10},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["l4", "l4", "l4", "l4", "l4_host", "l4_one", "run", "batch", "grad1", "gradn", "bath", "rk4"])
    dt = rng.choice([0.001, 0.002, 0.005, 0.01])
    if kind == "l4":
        d = rng.choice([2, 3, 4, 4, 6, 8])
        nt = _log(rng, 1500, {2: 200001, 3: 200001, 4: 200001, 6: 30000, 8: 16384}[d])
        tmax = min(nt - 1, _log(rng, 200, {2: 10000, 3: 10000, 4: 10000, 6: 3000, 8: 1000}[d]))
        return {"kind": kind, "h": "gue", "d": d, "ops": rng.choice([1, 1, 2]) if d < 6 else 1, "nt": nt, "dt": dt,
                "tmax": tmax, "tstep": rng.choice([1, 2, 3, 10]) if d < 6 else 4,
                "mode": rng.choice(["parity", "parity", "window"]),
                "phases": "cr" if d >= 6 else rng.choice(["libm", "libm", "cr"]), "scan": "bath"}
    if kind == "l4_host":
        nt = _log(rng, 1500, 200001)
        return {"kind": kind, "h": "gue", "d": rng.choice([2, 3]), "ops": 1, "nt": nt, "dt": dt,
                "tmax": min(nt - 1, _log(rng, 200, 10000)), "tstep": rng.choice([1, 3]), "scan": "bath"}
    if kind == "l4_one":
        nt = _log(rng, 500, 20000)
        return {"kind": kind, "h": "gue", "d": rng.choice([2, 3, 4]), "ops": 1, "nt": nt, "dt": dt,
                "t": rng.randrange(nt // 8, nt // 2), "scan": "system"}
    if kind == "run":
        d = rng.choice([2, 3, 4, 5])
        nt = _log(rng, 3000, 60000 if d < 5 else 8000)
        return {"kind": kind, "h": "gue", "d": d, "ops": 1, "nt": nt, "dt": dt,
                "steps": min(nt - 1, _log(rng, 200, 4000 if d < 5 else 1000)), "scan": "bath"}
    if kind == "batch":
        n = rng.randrange(4, 13)
        dims = [rng.choice([2, 2, 3, 3, 4]) for _ in range(n)]
        return {"kind": kind, "dims": " ".join(map(str, dims)),
                "log2nt": " ".join(str(rng.randrange(12, 18)) for _ in dims),
                "stride": " ".join(str(rng.choice([1, 2, 4, 8])) for _ in dims), "n_time": rng.randrange(100, 501),
                "dt": 0.005}
    if kind == "grad1":
        return {"kind": kind, "nt": 1 << rng.randrange(12, 17), "dt": 0.005, "steps": _log(rng, 300, 4000)}
    if kind == "gradn":
        spins = rng.choice([2, 3, 3, 4])
        return {"kind": kind, "spins": spins, "sets": rng.randrange(2, 9) if spins < 4 else rng.randrange(1, 4),
                "nt": 1 << rng.randrange(10, 13), "dt": 0.005, "steps": rng.randrange(50, 201)}
    if kind == "bath":
        return {"kind": kind, "nt": _log(rng, 2000, 200001), "dt": dt, "nf": rng.choice([3, 5, 7, 13])}
    D = rng.choice([4, 9, 16, 25, 36, 64])
    return {"kind": "rk4", "D": D, "steps": _log(rng, 200, 4000 if D <= 16 else 800), "dt": dt, "every": 10}


# --- inputs ---------------------------------------------------------------------


def _gue(d, r):
    M = (r.standard_normal((d, d)) + 1j * r.standard_normal((d, d))) / math.sqrt(2 * d)
    return np.tril(M, -1) + np.tril(M, -1).conj().T + np.diag(r.standard_normal(d) / math.sqrt(d))


def _model(h, d, ops, r):
    """Hamiltonian and coupling operators."""
    if h == "sx":
        return 0.5 * SX, [0.5 * SZ]
    if h == "spin_boson":
        return 0.5 * SZ + 0.5 * SX, [SZ.copy()]
    H = _gue(d, r)
    out = []
    for _ in range(ops):
        A = _gue(d, r)
        out.append(A / np.abs(np.linalg.eigvalsh(A)).max())
    return H, out


def _bath(r):
    """(kind, p0, p1, beta): Ohmic (0) or Drude-Lorentz (1)."""
    kind = int(r.integers(2))
    return kind, r.uniform(0.02, 0.2), r.uniform(2.0, 12.0), r.uniform(0.4, 3.0)


def _bath_obj(b):
    return taco.Ohmic(b[1], b[2]) if b[0] == 0 else taco.DrudeLorentz(b[1], b[2])


def _inputs(case, seed):
    """(H, ops, bath) of the cases that hold one system."""
    r = np.random.default_rng([7, int(seed)])
    hs = np.random.default_rng(11) if case["scan"] == "bath" else r
    H, ops = _model(case["h"], case["d"], case["ops"], hs)
    return H, ops, _bath(r)


def _batch_inputs(case, seed):
    r = np.random.default_rng([8, int(seed)])
    out = []
    for d, lg, s in zip(*(map(int, case[k].split()) for k in ("dims", "log2nt", "stride"))):
        H, ops = _model("gue", d, 1, r)
        n = case["n_time"]
        out.append((H, ops, _bath(r), 2 ** lg, [q * s for q in range(n)], n))
    return out


def _r0(N):
    r = np.zeros(N * N, complex)
    r[0] = 1.0
    return r


def _grad1_params(seed):
    r = np.random.default_rng([9, int(seed)])
    return np.array([0.05, 5.0, 1.0, 1.0, 1.0]) * r.uniform(0.8, 1.25, 5), r.uniform(0.95, 1.05, 5)


def _gradn_params(case, seed):
    r = np.random.default_rng([10, int(seed)])
    p = np.array([[0.05, 5.0, 1.0, 1.0, 1.0]] * case["sets"])
    p[:, :3] *= r.uniform(0.9, 1.1, (case["sets"], 3))
    p[:, 4] = r.uniform(0.5, 1.5, case["sets"])
    return p, r.uniform(0.95, 1.05, 5)


def _bath_omegas(case, seed):
    r = np.random.default_rng([12, int(seed)])
    b = _bath(r)
    w = np.sort(r.uniform(0.2, 4.0, case["nf"] // 2))
    return b, np.concatenate([-w[::-1], [0.0], w])


def _rk4_series(case, seed):
    """Slowly varying generators with decay: [steps + 1, D, D] and r0."""
    r = np.random.default_rng([13, int(seed)])
    D, n = case["D"], case["steps"] + 1
    A = _gue(D, r)
    G = (r.standard_normal((D, D)) + 1j * r.standard_normal((D, D))) / D
    s = np.exp(-np.arange(n) * case["dt"])[:, None, None]
    L = (-1j * A - 0.1 * np.eye(D))[None] + 0.1 * s * G[None]
    v = r.standard_normal(D) + 1j * r.standard_normal(D)
    return L, v / np.linalg.norm(v)


def _phases(case):
    return taco.phase_mode(taco.PHASE_CR if case.get("phases") == "cr" else taco.PHASE_LIBM)


def _gamma(system, b, nt, dt):
    return taco.bath_gamma_hip(nt - 1, dt, _bath_obj(b), b[3], system.omegas)[1]


def prepare(case, seed):
    k = case["kind"]
    s = dict(case)
    if k in ("l4", "l4_host", "l4_one", "run"):
        H, ops, b = _inputs(case, seed)
        s["system"] = taco.System.build(H, ops)
        with _phases(case):
            g = _gamma(s["system"], b, case["nt"], case["dt"])
        if k == "l4":
            s["dev"] = tcl4.DeviceSystem(s["system"], g)
        else:
            s["gamma"] = g
        if k in ("l4", "l4_host"):
            s["tidx"] = list(range(0, case["tmax"] + 1, case["tstep"]))
        s["r0"] = _r0(case["d"])
    elif k == "batch":
        with taco.phase_mode(taco.PHASE_CR):
            items = []
            for H, ops, b, nt, tidx, steps in _batch_inputs(case, seed):
                S = taco.System.build(H, ops)
                items.append(taco.BatchItem(S, _gamma(S, b, nt, case["dt"]), case["dt"], tidx, steps=steps,
                                            r0=_r0(S.N)))
            s["batch"] = taco.Batch(items)
        s["n"] = len(items)
    elif k == "grad1":
        s["prob"] = adjoint.SpinPairProblem(Nt=case["nt"], dt=case["dt"], steps=case["steps"])
        p, f = _grad1_params(seed)
        s["params"] = torch.tensor(p, dtype=torch.float64)
        with torch.no_grad():
            s["target"] = s["prob"].rho_lab(torch.tensor(p * f, dtype=torch.float64)).detach()
    elif k == "gradn":
        s["prob"] = adjoint.TfimChainProblem(n_spins=case["spins"], Nt=case["nt"], dt=case["dt"], steps=case["steps"])
        p, f = _gradn_params(case, seed)
        s["params"] = [torch.tensor(q, dtype=torch.float64) for q in p]
        with torch.no_grad(), taco.phase_mode(taco.PHASE_CR):
            s["targets"] = [s["prob"].rho_lab(q * torch.tensor(f)).detach() for q in s["params"]]
    elif k == "bath":
        s["bath"], s["omegas"] = _bath_omegas(case, seed)
    else:
        s["L"], s["r0"] = _rk4_series(case, seed)
    return s


def run(s):
    k = s["kind"]
    if k == "l4":
        with _phases(s), taco.fft_mode(taco.FFT_WINDOW if s["mode"] == "window" else taco.FFT_PARITY):
            return tcl4.build_l4_dev(s["dev"], s["dt"], s["tidx"])
    if k == "l4_host":
        return taco.build_TCL4_generator_hip_fused_batch(s["system"], s["gamma"], s["dt"], s["tidx"])
    if k == "l4_one":
        return taco.build_TCL4_generator_hip_fused(s["system"], s["gamma"], s["dt"], s["t"])
    if k == "run":
        return taco.tcl4_propagate(s["system"], s["gamma"], s["dt"], s["steps"], s["r0"])
    if k == "batch":
        with taco.phase_mode(taco.PHASE_CR):
            b = s["batch"].run(graph=True)
        return [{"l4": b.l4(q), "rho": b.rho(q)} for q in range(s["n"])]
    if k == "grad1":
        p = s["params"].clone().requires_grad_(True)
        loss = s["prob"].loss(p, s["target"])
        (g,) = torch.autograd.grad(loss, p)
        return {"loss": loss.detach(), "grad": g}
    if k == "gradn":
        with taco.phase_mode(taco.PHASE_CR):
            ps = [p.clone().requires_grad_(True) for p in s["params"]]
            losses = s["prob"].losses_many(ps, s["targets"])
            gs = torch.autograd.grad(sum(losses), ps)
        return {"loss": torch.stack([x.detach() for x in losses]), "grad": torch.stack(gs)}
    if k == "bath":
        C, G = taco.bath_gamma_hip(s["nt"] - 1, s["dt"], _bath_obj(s["bath"]), s["bath"][3], s["omegas"])
        return {"C": C, "gamma": G}
    seen = []
    r = taco.propagate_rk4_dense(s["L"], s["r0"], 0.0, s["dt"], on_sample=lambda t, v: seen.append(v),
                                 sample_every=s["every"])
    return {"r": r, "samples": np.stack(seen)}


# --- what a pass cannot do without ------------------------------------------------


def _l4_work(d, nf, nt, T, npos, ops=1):
    """The Gamma rows below T read, L4 written; the causal convolutions of the
    triples L4 reads (F: about d^4 patterns, C: d^2 (2 d - 1) outer pairs
    below nf^2, any middle bucket) by FFTs of the window's length, one input
    transform per two of them, and the L4 contractions."""
    n = 1 << max(1, (2 * T - 2).bit_length())
    paths = min(nf ** 3, 2 * d ** 4) + min(nf * nf, 2 * d ** 3) * nf
    fft = 5.0 * n * math.log2(n)
    l4 = 8.0 * (4 * d ** 3 * nf + 2 * d ** 4 + 2 * d ** 5 + d ** 3 * nf) * ops * ops
    return {"bytes": 16.0 * (nf * T + npos * d ** 4), "flops": 1.5 * paths * fft + npos * l4}


def _nf(h, d):
    return 3 if d == 2 else d * d - d + 1


def work(case):
    k = case["kind"]
    if k in ("l4", "l4_host"):
        w = _l4_work(case["d"], _nf(case["h"], case["d"]), case["nt"], case["tmax"] + 1,
                     case["tmax"] // case["tstep"] + 1, case["ops"])
        return w
    if k == "l4_one":
        return _l4_work(case["d"], _nf(case["h"], case["d"]), case["nt"], case["t"] + 1, 1)
    if k == "run":
        d, n = case["d"], case["steps"] + 1
        w = _l4_work(d, _nf(case["h"], d), case["nt"], n, n)
        return {"bytes": w["bytes"], "flops": w["flops"] + n * 32.0 * d ** 4}
    if k == "batch":
        tot = {"bytes": 0.0, "flops": 0.0}
        for d, lg, s in zip(*(map(int, case[q].split()) for q in ("dims", "log2nt", "stride"))):
            n = case["n_time"]
            w = _l4_work(d, _nf("gue", d), 2 ** lg, n * s, 2 * n)
            tot["bytes"] += w["bytes"]
            tot["flops"] += w["flops"] + n * 32.0 * d ** 4
        return tot
    if k in ("grad1", "gradn"):
        # forward and a reverse of twice its operations
        if k == "grad1":
            d, nf, sets = 4, 5, 1
        else:
            d, nf, sets = 2 ** case["spins"], {2: 9, 3: 31, 4: 81}[case["spins"]], case["sets"]
        n = case["steps"] + 1
        w = _l4_work(d, nf, case["nt"], n, n)
        return {"bytes": sets * 3.0 * w["bytes"], "flops": sets * 3.0 * (w["flops"] + n * 32.0 * d ** 4)}
    if k == "bath":
        n = 1 << (2 * case["nt"] - 1).bit_length()
        return {"bytes": 16.0 * case["nt"] * (1 + case["nf"]),
                "flops": 5.0 * n * math.log2(n) + 24.0 * case["nt"] * case["nf"]}
    D, n = case["D"], case["steps"]
    return {"bytes": 16.0 * (D * D * (n + 1) + D * (n // case["every"] + 2)), "flops": n * 4 * 8.0 * D * D}


# --- the same in plain torch, 64 bits ----------------------------------------------


def _dev():
    return torch.device("cuda") if torch.cuda.is_available() else torch.device("cpu")


def _x_system(H, ops, tol=1e-9):
    """Eigenbasis (each vector's largest entry real positive), coupling
    operators in it, bucket frequencies, mirror and pair map."""
    e, U = np.linalg.eigh(H)
    N = e.size
    for c in range(N):
        m = np.abs(U[:, c])
        best = 0
        for q in range(1, N):
            if m[q] > m[best] + 1e-12:
                best = q
        U[:, c] *= U[best, c].conj() / m[best]
    reps, p2f = [], np.zeros((N, N), int)
    for a in range(N):
        for b in range(N):
            w = e[a] - e[b]
            q = next((i for i, v in enumerate(reps) if abs(v - w) <= tol), None)
            if q is None:
                q = len(reps)
                reps.append(w)
            p2f[a, b] = q
    perm = np.argsort(reps)
    om = np.array(reps)[perm]
    mirror = np.array([int(np.argmin(np.abs(om + w))) for w in om])
    dev = _dev()
    return (torch.tensor(e, device=dev), [torch.tensor(U.conj().T @ A @ U, device=dev) for A in ops],
            torch.tensor(om, device=dev), torch.tensor(mirror, device=dev),
            torch.tensor(np.argsort(perm)[p2f], device=dev))


def _x_bath(kind, p0, p1, beta, nt, dt):
    """C(t_n), n < nt: the FFT of the sampled spectrum."""
    n = 1 << (2 * nt - 1).bit_length()
    dw, wny = 2.0 * math.pi / (dt * n), math.pi / dt

    def J(w):
        return p0 * w * torch.exp(-w / p1) if kind == 0 else 2.0 * p0 * p1 * w / (w * w + p1 * p1)

    k = torch.arange(1, n // 2, device=_dev(), dtype=torch.float64)
    kms = torch.exp(-beta * dw * k)
    sp = (math.pi / 2) * J(dw * k) / (1.0 - kms)
    one = torch.ones(1, dtype=torch.float64, device=_dev())
    r = torch.exp(-beta * dw * one)
    s0 = 0.5 * (math.pi / 2) * J(dw * one) * (1.0 + r) / (1.0 - r)
    x = torch.exp(-beta * wny * one)
    sny = 0.25 * math.pi * J(wny * one) * (1.0 + 2.0 * x / (1.0 - x))
    S = torch.cat([s0, sp, sny, (sp * kms).flip(0)])
    return (dw / math.pi) * torch.fft.fft(S.to(torch.complex128))[:nt]


def _x_gamma(C, om, dt, T):
    """Trapezoid prefix integrals of e^{i w t} C(t), [nf, T]."""
    t = torch.arange(T, device=C.device, dtype=torch.float64) * dt
    y = torch.exp(1j * om[:, None] * t[None]) * C[None, :T]
    z = torch.zeros((om.numel(), 1), dtype=y.dtype, device=y.device)
    return torch.cat([z, (dt / 2) * torch.cumsum(y[:, :-1] + y[:, 1:], 1)], 1)


def _x_fcr(g, om, mirror, dt, pos):
    """F, C, R [nf, nf, nf, len(pos)] at the times pos from g [nf, T]."""
    nf, T = g.shape
    n = 1 << max(1, (2 * T - 2).bit_length())
    t = torch.arange(T, device=g.device, dtype=torch.float64) * dt
    out = ([], [], [])
    h = [torch.fft.fft(g[mirror], n), torch.fft.fft(g.conj(), n)]
    for i in range(nf):
        row = ([], [], [])
        for j in range(nf):
            w = om[i] + om[j] + om  # [k]
            pm = torch.exp(-1j * w[:, None] * t[None])
            a = g[i][None] * pm
            fa = torch.fft.fft(a, n)
            for q, g2 in ((0, g[mirror[j]]), (1, g[j].conj())):
                conv = torch.fft.ifft(fa * h[q][j][None], n)[:, :T]
                row[q].append((dt * (a * torch.cumsum(g2[None] * pm.conj(), 1) - conv))[:, pos])
            row[2].append((dt * (g[i][None] * torch.cumsum(g[j][None] * pm, 1)
                                 - torch.cumsum((g[i] * g[j])[None] * pm, 1)))[:, pos])
        for q in range(3):
            out[q].append(torch.stack(row[q]))
    return [torch.stack(v) for v in out]


def _x_l4(F, C, R, f, ops):
    """L4 [N, N, N, N, t] indexed (n, m, i, j) from the slices."""
    N = f.shape[0]
    q = torch.arange(N, device=f.device)
    n_, a_, b_, i_ = q[:, None, None, None], q[None, :, None, None], q[None, None, :, None], q[None, None, None, :]
    x, y, z = q[:, None, None], q[None, :, None], q[None, None, :]
    Xp = (C + R).permute(0, 2, 1, 3)  # [outer, outer, middle, t]
    XA, XB = Xp[f[y, x], f[x, z]], Xp[f[z, y], f[x, z]]  # (a, b, i, g, t)
    M = F[f[b_, a_], f[b_, i_], f[n_, b_]] - R[f[b_, a_], f[n_, a_], f[a_, i_]]
    I = F[f[a_, n_], f[b_, i_], f[n_, b_]]
    K = R[f[i_, b_], f[n_, a_], f[a_, i_]]
    T = 0
    eye = torch.eye(N, dtype=F.dtype, device=F.device)
    for A in ops:
        for B in ops:
            Q = torch.einsum("ab,bi,abigt->aigt", A, B, XA) - torch.einsum("ab,bi,abigt->aigt", B, A, XB)
            S = (torch.einsum("na,ab,bi,nabit->nit", A, B, B, I) - torch.einsum("na,ab,bi,nabit->nit", B, A, B, M)
                 - torch.einsum("na,ab,bi,nabit->nit", B, B, A, K))
            S67 = torch.einsum("na,aigt->nigt", A, Q)
            D = -torch.einsum("na,ait->nit", A, S)
            T = (T + torch.einsum("jm,nit->nimjt", A, S) + torch.einsum("jm,nijmt->nimjt", B, S67[:, :, f])
                 - torch.einsum("jb,bm,nijbt->nimjt", B, A, Q[:, :, f]) + torch.einsum("jm,nit->nimjt", eye, D))
    return T.permute(0, 2, 1, 3, 4) + T.permute(2, 0, 3, 1, 4).conj()  # (n, m, i, j): T(n,i;m,j) + conj T(m,j;n,i)


def _x_rows(L):
    """[t, row, col] with row = n + m N, col = i + j N."""
    N, nt = L.shape[0], L.shape[-1]
    return L.permute(4, 1, 0, 3, 2).reshape(nt, N * N, N * N)


def _x_tcl2(g, e, f, ops):
    """The second-order generator at every column of g [nf, t]: [t, N^2, N^2]."""
    N, nf = f.shape[0], g.shape[0]
    eye = torch.eye(N, dtype=torch.complex128, device=g.device)
    mask = (f[None] == torch.arange(nf, device=f.device)[:, None, None]).to(torch.complex128)
    H = torch.diag(e).to(torch.complex128)[None]
    L = 0
    gam, lamb = (2.0 * g.real).to(torch.complex128), g.imag.to(torch.complex128)
    for A in ops:
        P = mask * A[None]
        AA = torch.einsum("bqr,bqc->brc", P.conj(), P)
        H = H + torch.einsum("bt,brc->trc", lamb, AA)
        G = torch.einsum("bt,brc->trc", gam, AA)
        L = (L + torch.einsum("bt,bxy,buv->txuyv", gam, P.conj(), P)
             - 0.5 * torch.einsum("xy,tuv->txuyv", eye, G) - 0.5 * torch.einsum("uv,tyx->txuyv", eye, G))
    L = L - 1j * (torch.einsum("xy,tuv->txuyv", eye, H) - torch.einsum("uv,tyx->txuyv", eye, H))
    return L.reshape(g.shape[1], N * N, N * N)


def _x_rk4(L, r, dt):
    out = [r]
    Lh = 0.5 * (L[:-1] + L[1:])
    for L0, L1, Lm in zip(L[:-1].unbind(0), L[1:].unbind(0), Lh.unbind(0)):
        k1 = L0 @ r
        k2 = Lm @ (r + (0.5 * dt) * k1)
        k3 = Lm @ (r + (0.5 * dt) * k2)
        k4 = L1 @ (r + dt * k3)
        r = r + (dt / 6.0) * (k1 + 2.0 * k2 + 2.0 * k3 + k4)
        out.append(r)
    return torch.stack(out)


def _x_gen(C, e, ops, om, mirror, f, dt, pos):
    """L4 rows at the times pos, and Gamma up to the last of them."""
    g = _x_gamma(C, om, dt, int(pos[-1]) + 1)
    return _x_rows(_x_l4(*_x_fcr(g, om, mirror, dt, torch.as_tensor(pos, device=g.device)), f, ops)), g


def _x_states(C, e, ops, om, mirror, f, dt, steps):
    L, g = _x_gen(C, e, ops, om, mirror, f, dt, range(steps + 1))
    r = torch.zeros(f.shape[0] ** 2, dtype=torch.complex128, device=g.device)
    r[0] = 1.0
    return _x_rk4(L + _x_tcl2(g, e, f, ops), r, dt)


def _x_pair(p, nt, dt, steps):
    """rho_lab(t) of the spin pair as a differentiable function of
    p = (alpha, omega_c, beta, eps, delta)."""
    dev = _dev()
    sz, sx = torch.tensor(SZ.real, device=dev), torch.tensor(SX.real, device=dev)
    e1, u = torch.linalg.eigh(0.5 * p[3] * sz + 0.5 * p[4] * sx)
    e = (e1[:, None] + e1[None]).reshape(-1)
    U = torch.kron(u, u).to(torch.complex128)
    i2 = torch.eye(2, dtype=torch.float64, device=dev)
    A = torch.kron(sz, i2) + torch.kron(i2, sz)
    om = (e1[1] - e1[0]) * torch.tensor([-2.0, -1.0, 0.0, 1.0, 2.0], dtype=torch.float64, device=dev)
    up = torch.tensor([0, 1, 1, 2], device=dev)
    f = up[:, None] - up[None] + 2
    C = _x_bath(0, p[0], p[1], p[2], nt, dt)
    r = _x_states(C, e, [U.conj().T @ A.to(torch.complex128) @ U], om, torch.arange(4, -1, -1, device=dev), f, dt, steps)
    return U @ r.reshape(-1, 4, 4).transpose(1, 2) @ U.conj().T


def _np(x):
    return x.detach().cpu().numpy()


def exact(case, seed):
    k = case["kind"]
    dt = case["dt"]
    if k in ("l4", "l4_host", "l4_one", "run"):
        H, ops, b = _inputs(case, seed)
        S = _x_system(H, ops)
        C = _x_bath(*b, case["nt"], dt)
        if k == "run":
            return _np(_x_states(C, *S, dt, case["steps"]))
        pos = [case["t"]] if k == "l4_one" else range(0, case["tmax"] + 1, case["tstep"])
        L = _x_gen(C, *S, dt, pos)[0]
        if k == "l4":  # column-major blocks
            return _np(L.transpose(1, 2).reshape(L.shape[0], -1))
        return _np(L[0] if k == "l4_one" else L)
    if k == "batch":
        out = []
        for H, ops, b, nt, tidx, steps in _batch_inputs(case, seed):
            S = _x_system(H, ops)
            C = _x_bath(*b, nt, dt)
            out.append({"l4": _np(_x_gen(C, *S, dt, tidx)[0]), "rho": _np(_x_states(C, *S, dt, steps))})
        return out
    if k == "grad1":
        p, f = _grad1_params(seed)
        with torch.no_grad():
            target = _x_pair(torch.tensor(p * f, device=_dev()), case["nt"], dt, case["steps"])
        p = torch.tensor(p, device=_dev(), requires_grad=True)
        d = _x_pair(p, case["nt"], dt, case["steps"]) - target
        loss = (d.real ** 2 + d.imag ** 2).sum()
        (g,) = torch.autograd.grad(loss, p)
        return {"loss": loss.detach().cpu(), "grad": g.cpu()}
    if k == "gradn":
        return None  # the chain's L4 in plain torch, forward and back, takes far over 20 seconds
    if k == "bath":
        b, om = _bath_omegas(case, seed)
        C = _x_bath(*b, case["nt"], dt)
        return {"C": _np(C), "gamma": _np(_x_gamma(C, torch.tensor(om, device=_dev()), dt, case["nt"]).T)}
    L, r = _rk4_series(case, seed)
    s = _np(_x_rk4(torch.tensor(L), torch.tensor(r), dt))
    at = list(range(0, case["steps"], case["every"])) + [case["steps"]]
    return {"r": s[-1], "samples": s[at]}
