"""The work that a user of netket_amd has it do, as cases that can be timed and compared.

A case names one path of the VMC step and its sizes:

* ``step``    whole optimisation steps: ``driver.run(1)`` of ``VMC`` with the SR preconditioner or
              of ``VMC_SR`` (SR, or minSR where there are more parameters than samples);
* ``sample``  ``MCState.sample``: reset, discarded and kept Metropolis sweeps;
* ``eloc``    ``MCState.local_estimators`` on samples in hand;
* ``qgt``     ``QGTJacobianDense(...).to_dense()`` on samples in hand;
* ``solve``   ``solver.cholesky`` of a dense FP64 system.

Models are RBMs in both parameter types (FP64 is what a program gets that does not ask for a type)
and the two-layer network; Hamiltonians the transverse-field Ising model (``tfim``), the Heisenberg
chain (``heisenberg``) and the J1-J2 model (``j1j2``).  Weights are normal with a spread that gives
log-amplitude differences of order one, as part way through an optimisation.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import netket_amd as nk
from netket_amd.optimizer import solver


def listed():
    return [
        # The first tutorial-sized problem: a 16-site chain with NetKet's default 16 chains and about
        # 1000 samples; launches and host work are all that count.
        dict(name="step_tfim16_f64", path="step", ham="tfim", dim=1, L=16, h=1.0, model="rbm", alpha=1,
             f64=True, chains=16, samples=1008, discard=16, precond=True),
        # The benchmark's step: Heisenberg L=64, FP32 RBM alpha=2, dense S (8384^2) and Cholesky.
        dict(name="step_heis64_f32", path="step", ham="heisenberg", dim=1, L=64, h=0.0, model="rbm", alpha=2,
             f64=False, chains=4096, samples=16384, discard=5, precond=False),
        # A large job of the serving stream: 12x12 lattice, alpha=4, 8192 samples, minSR.
        dict(name="step_tfim12x12_f32", path="step", ham="tfim", dim=2, L=12, h=1.5, model="rbm", alpha=4,
             f64=False, chains=1024, samples=8192, discard=5, precond=False),
        # The sampler of the benchmark's workload in the default parameter type, exchange moves.
        dict(name="sample_heis64_f64", path="sample", ham="heisenberg", dim=1, L=64, h=0.0, model="rbm", alpha=2,
             f64=True, chains=4096, samples=16384, discard=5),
        # The sampler of the 20x20 lattice with 3200 hidden units (W beyond LDS), local moves.
        dict(name="sample_tfim20x20_f32", path="sample", ham="tfim", dim=2, L=20, h=3.04, model="rbm", alpha=8,
             f64=False, chains=8192, samples=32768, discard=5),
        # The network's sampler on the J1-J2 lattice, exchange moves over two bond lengths.
        dict(name="sample_j1j2_ffnn_f32", path="sample", ham="j1j2", dim=2, L=10, h=0.0, model="ffnn", alpha=0,
             h1=400, h2=400, f64=False, chains=8192, samples=16384, discard=5),
        # Local energies: the chain in the default type, the wide RBM, and the network with up to 400
        # connected configurations per sample.
        dict(name="eloc_heis64_f64", path="eloc", ham="heisenberg", dim=1, L=64, h=0.0, model="rbm", alpha=2,
             f64=True, chains=4096, samples=16384),
        dict(name="eloc_tfim20x20_f32", path="eloc", ham="tfim", dim=2, L=20, h=3.04, model="rbm", alpha=8,
             f64=False, chains=8192, samples=32768),
        dict(name="eloc_j1j2_ffnn_f32", path="eloc", ham="j1j2", dim=2, L=10, h=0.0, model="ffnn", alpha=0,
             h1=400, h2=400, f64=False, chains=8192, samples=16384),
        # The dense S of the benchmark's workload in the default parameter type.
        dict(name="qgt_heis64_f64", path="qgt", ham="heisenberg", dim=1, L=64, h=0.0, model="rbm", alpha=2,
             f64=True, chains=4096, samples=16384),
        # The solve alone: a small SR system (40-site chain, alpha=1) and the minSR system of the 20x20 lattice.
        dict(name="solve_1680", path="solve", n=1680, rank=1024, shift=0.01),
        dict(name="solve_32768", path="solve", n=32768, rank=3600, shift=0.01),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["step", "sample", "eloc", "qgt", "solve", "solve"])
    if path == "solve":
        n = _log_int(rng, 33, 16384)
        return dict(path="solve", n=n, rank=max(8, int(n * rng.uniform(0.3, 1.0))), shift=rng.choice([1e-3, 1e-2]))
    f64 = rng.random() < 0.5
    ham = rng.choice(["tfim", "tfim", "heisenberg", "j1j2"] if path in ("sample", "eloc") else ["tfim", "heisenberg"])
    c = dict(path=path, ham=ham, h=round(rng.uniform(0.5, 3.0), 2), model="rbm", f64=f64)
    if ham == "tfim" and rng.random() < 0.5:
        c.update(dim=2, L=rng.randint(4, 8 if path in ("step", "qgt") else 12 if f64 else 20))
    elif ham == "j1j2":
        c.update(dim=2, L=rng.choice([4, 6, 8, 10]))
    else:
        c.update(dim=1, L=_log_int(rng, 8, 64 if path in ("step", "qgt") else 128))
        if ham == "heisenberg":
            c["L"] += c["L"] % 2
    n = c["L"] ** c["dim"]
    c["alpha"] = rng.choice([1, 2] if path in ("step", "qgt") or n > 144 else [1, 2, 4])
    if ham == "j1j2" and rng.random() < 0.7:
        c.update(model="ffnn", alpha=0, f64=False, h1=rng.randint(24, 400), h2=rng.randint(24, 400))
    chains = _log_int(rng, 16, 4096)
    length = max(1, min(_log_int(rng, 1, 64), 16384 // chains))
    c.update(chains=chains, samples=chains * length)
    if path in ("step", "sample"):
        c["discard"] = rng.choice([0, 2, 5])
    if path == "step":
        c["precond"] = rng.random() < 0.3
    return c


# ---------------------------------------------------------------------------
# what a program has in hand
# ---------------------------------------------------------------------------
def _n_sites(c):
    return c["L"] ** c["dim"]


def _system(c):
    """(Hamiltonian, sampler) of a case."""
    order = 2 if c["ham"] == "j1j2" else 1
    g = nk.graph.Square(c["L"], max_neighbor_order=order) if c["dim"] == 2 else nk.graph.Chain(c["L"])
    if c["ham"] == "tfim":
        hi = nk.hilbert.Spin(0.5, N=g.n_nodes)
        return nk.operator.Ising(hi, g, h=c["h"], J=1.0), nk.sampler.MetropolisLocal(hi, n_chains=c["chains"])
    hi = nk.hilbert.Spin(0.5, N=g.n_nodes, total_sz=0)
    if c["ham"] == "j1j2":
        H = nk.operator.Heisenberg(hi, g, J=[1.0, 0.5], sign_rule=[False, False])
    else:
        H = nk.operator.Heisenberg(hi, g)
    return H, nk.sampler.MetropolisExchange(hi, graph=g, n_chains=c["chains"])


def _blocks(c):
    """Sizes of the parameter blocks in ravel order, and the spread of each."""
    n = _n_sites(c)
    if c["model"] == "ffnn":
        h1, h2 = c["h1"], c["h2"]
        return [(h1, 0.1), (n * h1, 0.5 / math.sqrt(n)), (h2, 0.1), (h1 * h2, 0.5 / math.sqrt(h1))]
    m = c["alpha"] * n
    return [(m, 0.05), (n * m, 0.6 / math.sqrt(m)), (n, 0.05)]


def _dtype(c):
    return torch.float64 if c["f64"] else torch.float32


def _inputs(c, seed):
    """(flat parameters, configurations of shape (chains, length, sites)) of a seed."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    flat = torch.cat([s * torch.randn(k, generator=gen, device="cuda", dtype=torch.float64) for k, s in _blocks(c)])
    n = _n_sites(c)
    r = torch.rand((c["samples"], n), generator=gen, device="cuda")
    if c["ham"] == "tfim":
        x = torch.where(r < 0.5, 1, -1)
    else:
        x = torch.where(r.argsort(dim=1) < n // 2, 1, -1)
    return flat.to(_dtype(c)), x.to(torch.int8).reshape(c["chains"], -1, n)


def _matrix(c, seed):
    """An SR or minSR system: X X^T / r + shift I of r samples whose modes fall off, and its right-hand side."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    n, r = c["n"], c["rank"]
    x = torch.randn((n, r), generator=gen, device="cuda", dtype=torch.float64)
    x *= (torch.arange(1, r + 1, device="cuda", dtype=torch.float64) ** -0.5)
    a = x @ x.T
    a.diagonal().add_(c["shift"])
    return a, torch.randn(n, generator=gen, device="cuda", dtype=torch.float64)


def prepare(case, seed):
    c = dict(case)
    if c["path"] == "solve":
        a, b = _matrix(c, seed)
        return dict(path="solve", a=a, b=b)
    H, sa = _system(c)
    dt = np.float64 if c["f64"] else np.float32
    if c["model"] == "ffnn":
        model = nk.models.FFNN(hidden_dims=(c["h1"], c["h2"]), param_dtype=dt)
    else:
        model = nk.models.RBM(alpha=c["alpha"], param_dtype=dt)
    vs = nk.vqs.MCState(sa, model, n_samples=c["samples"], n_discard_per_chain=c.get("discard", 5), seed=int(seed))
    flat, x = _inputs(c, seed)
    vs.parameters = flat
    st = dict(path=c["path"], vs=vs, H=H)
    if c["path"] in ("eloc", "qgt"):
        vs._samples = x
    if c["path"] == "step":
        opt = nk.optimizer.Sgd(0.002)
        if c["precond"]:
            sr = nk.optimizer.SR(nk.optimizer.QGTJacobianDense, solver=solver.cholesky, diag_shift=0.01)
            st["driver"] = nk.VMC(H, opt, variational_state=vs, preconditioner=sr)
        else:
            st["driver"] = nk.VMC_SR(H, opt, diag_shift=0.01, variational_state=vs, linear_solver=solver.cholesky)
    return st


def run(state):
    if state["path"] == "solve":
        return {"x": solver.cholesky(state["a"], state["b"])[0]}
    vs = state["vs"]
    if state["path"] == "sample":
        x = vs.sample()
        s = vs.sampler_state
        return {"samples": x, "log_prob": s.log_prob, "accepted": s.n_accepted_proc}
    if state["path"] == "eloc":
        return {"eloc": vs.local_estimators(state["H"])}
    if state["path"] == "qgt":
        return {"S": nk.optimizer.QGTJacobianDense(vs, diag_shift=0.01).to_dense()}
    state["driver"].run(1)
    return {"parameters": vs.parameters_flat}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _sizes(c):
    n = _n_sites(c)
    n_par = sum(k for k, _ in _blocks(c))
    w = 8 if c["f64"] else 4
    hidden = c["h1"] + c["h2"] if c["model"] == "ffnn" else c["alpha"] * n
    # one log-amplitude from its neighbour's: a few rows of the first layer, the activations, the second layer
    amp = 12.0 * hidden + (2.0 * c["h1"] * c["h2"] if c["model"] == "ffnn" else 0.0)
    return n, n_par, w, hidden, amp


def work(case):
    c = dict(case)
    if c["path"] == "solve":
        n = float(c["n"])
        return {"bytes": 8 * n * n + 16 * n, "flops": n**3 / 3 + 2 * n * n}
    n, n_par, w, hidden, amp = _sizes(c)
    ns = c["samples"]
    sweeps = c["chains"] * c.get("discard", 0) + ns
    sample = {"bytes": w * n_par + n * (2 * c["chains"] + ns) + 2.0 * c["chains"] * (w + 8), "flops": sweeps * n * amp}
    bonds = {"tfim": n, "heisenberg": n / 2, "j1j2": 2 * n}[c["ham"]]
    eloc = {"bytes": w * n_par + ns * (n + 8.0), "flops": ns * (bonds * amp + 2.0 * n * hidden)}
    if c["path"] == "sample":
        return sample
    if c["path"] == "eloc":
        return eloc
    gram = {"bytes": w * n_par + ns * n + 8.0 * n_par * n_par, "flops": 1.0 * ns * n_par * n_par}
    if c["path"] == "qgt":
        return gram
    if n_par > ns and not c["precond"]:
        gram = {"bytes": 8.0 * ns * ns, "flops": 1.0 * ns * ns * (hidden + n)}
    k = float(min(n_par, ns) if not c["precond"] else n_par)
    return {"bytes": sample["bytes"] + 2 * w * n_par, "flops": sample["flops"] + eloc["flops"] + gram["flops"] + k**3 / 3}


# ---------------------------------------------------------------------------
# what a pass returns, in 64 bits
# ---------------------------------------------------------------------------
def _log_cosh(x):
    a = x.abs()
    return a + torch.log1p(torch.exp(-2 * a)) - math.log(2.0)


def _first_layer(c, p, x):
    """Pre-activations of the first layer for configurations x (rows, sites)."""
    return x @ p[1].reshape(_n_sites(c), -1) + p[0]


def _log_psi(c, p, x, th):
    """log psi of configurations x (rows, sites) with first-layer pre-activations th."""
    if c["model"] == "ffnn":
        return _log_cosh(_log_cosh(th) @ p[3].reshape(c["h1"], -1) + p[2]).sum(-1)
    return _log_cosh(th).sum(-1) + x @ p[2]


def _bonds(c):
    """(site, site, coupling) of every bond of the periodic lattice."""
    if c["dim"] == 1:
        ls = [((i,), ((i + 1) % c["L"],)) for i in range(c["L"])]
        js = [1.0] * len(ls)
        flat = [(a[0], b[0]) for a, b in ls]
    else:
        k, flat, js = c["L"], [], []
        steps = [(0, 1, 1.0), (1, 0, 1.0)] + ([(1, 1, 0.5), (1, -1, 0.5)] if c["ham"] == "j1j2" else [])
        for i in range(k):
            for j in range(k):
                for di, dj, v in steps:
                    flat.append((i * k + j, ((i + di) % k) * k + (j + dj) % k))
                    js.append(v)
    seen = {}
    for (a, b), v in zip(flat, js):
        seen.setdefault((min(a, b), max(a, b)), v)
    return [(a, b, v) for (a, b), v in seen.items()]


def _local_energies(c, p, x):
    """E_loc of configurations x (rows, sites)."""
    th, w = _first_layer(c, p, x), p[1].reshape(x.shape[1], -1)
    lp = _log_psi(c, p, x, th)
    bonds = _bonds(c)
    a = torch.tensor([b[0] for b in bonds], device=x.device)
    b = torch.tensor([b[1] for b in bonds], device=x.device)
    v = torch.tensor([b[2] for b in bonds], device=x.device, dtype=x.dtype)
    e = ((x[:, a] * x[:, b]) * v).sum(-1)
    if c["ham"] == "tfim":
        moves = [(i,) for i in range(x.shape[1])]
    else:
        moves = [(i, j) for i, j, _ in bonds]
    sign = -1.0 if c["ham"] == "heisenberg" else 1.0  # the sign rule, on by default where it can be
    for k, sites in enumerate(moves):
        rows = slice(None) if len(sites) == 1 else torch.nonzero(x[:, sites[0]] * x[:, sites[1]] < 0)[:, 0]
        y, ty = x[rows].clone(), th[rows].clone()
        for i in sites:  # a flip, or an exchange of two different spins
            ty -= 2 * y[:, i:i + 1] * w[i]
            y[:, i] *= -1
        mel = -c["h"] if len(sites) == 1 else sign * 2.0 * bonds[k][2]
        e[rows] += mel * torch.exp(_log_psi(c, p, y, ty) - lp[rows])
    return e


def exact(case, seed):
    c = dict(case)
    if c["path"] == "solve":
        a, b = _matrix(c, seed)
        return {"x": torch.cholesky_solve(b[:, None], torch.linalg.cholesky(a))[:, 0]}
    if c["path"] not in ("eloc", "qgt"):
        return None  # chains follow the sampler's own random stream
    flat, x = _inputs(c, seed)
    p = torch.split(flat.double(), [k for k, _ in _blocks(c)])
    n, n_par, _, hidden, _ = _sizes(c)
    xs = x.reshape(-1, n)
    if c["path"] == "eloc":
        rows = 16384 if hidden < 1024 else 4096
        return {"eloc": torch.cat([_local_energies(c, p, q.double()) for q in xs.split(rows)]).reshape(c["chains"], -1)}
    s, mean = torch.zeros((n_par, n_par), dtype=torch.float64, device="cuda"), 0.0
    parts = []
    for q in xs.split(4096):
        q = q.double()
        t = torch.tanh(_first_layer(c, p, q))
        parts.append(torch.cat([t, (q[:, :, None] * t[:, None, :]).flatten(1), q], dim=1))
        mean = mean + parts[-1].sum(0) / c["samples"]
    for o in parts:
        o -= mean
        s.addmm_(o.T.contiguous(), o, alpha=1.0 / c["samples"])
    s.diagonal().add_(0.01)
    return {"S": s}
