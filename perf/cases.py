"""Work that users of this package have it do, each through its public entry
points: whole simulations of the four library programs (with the model reset
to its seed, as replicate studies and calibrations run them), the gradient of
the differentiable one, a generic model written against the agent API, and a
trace of requests through the batching server.

A case is a dict of plain values; ``kind`` names the program.  ``mode`` is the
random stream layout (1: JAX's partitionable default, 0: the original one).
"""
import contextlib
import io
import math

import numpy as np
import torch

import jaxabm_amd as J
from jaxabm_amd import numpy as jnp
from jaxabm_amd import random as jr


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest calls: a classroom-size wealth run, latency and launches
        dict(name="wealth_64x20", kind="wealth", n=64, steps=20, mode=1),
        # the README's wealth run, one workgroup
        dict(name="wealth_1000x100", kind="wealth", n=1000, steps=100, mode=1),
        # the middle of the one-workgroup range, odd size, original stream
        dict(name="wealth_5003x150", kind="wealth", n=5003, steps=150, mode=0),
        # the largest wealth request of the serving trace, run alone
        dict(name="wealth_247720x229", kind="wealth", n=247_720, steps=229, mode=1),
        # an epidemic on a town-size network, original stream
        dict(name="sir_20011x160", kind="sir", n=20_011, m=3, steps=160, beta=0.08, gamma=0.1,
             infected=20, mode=0),
        # the headline epidemic: one million agents, a year of days
        dict(name="sir_1Mx365", kind="sir", n=1_000_000, m=4, steps=365, beta=0.05, gamma=0.1,
             infected=100, mode=1),
        # a small ragged segregation grid
        dict(name="schelling_61x90x80", kind="schelling", h=61, w=90, steps=80, mode=0),
        # the benchmark's segregation grid
        dict(name="schelling_512x512x200", kind="schelling", h=512, w=512, steps=200, mode=1),
        # a calibrator's small population: loss and gradient of 12 candidates
        dict(name="deffuant_1001x12x60", kind="deffuant", n=1001, batch=12, steps=60, ckpt=10,
             grad=True, mode=1),
        # the benchmark's gradient evaluation: a 256-instance parameter sweep
        dict(name="deffuant_65536x256x200", kind="deffuant", n=65_536, batch=256, steps=200,
             ckpt=20, grad=True, mode=1),
        # a model with no library kernel, built and run as graph replays
        dict(name="generic_10000x200", kind="generic", n=10_000, steps=200),
        # uneven requests through the continuous-batching server
        dict(name="serving_48", kind="serving", requests=48, n_min=1000, n_max=256_000),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["wealth", "wealth", "wealth", "sir", "sir", "schelling", "schelling",
                       "deffuant", "deffuant", "deffuant", "generic", "serving"])
    mode = 0 if rng.random() < 0.25 else 1
    if kind == "wealth":
        n = _log(rng, 20, 240_000)
        return dict(kind=kind, n=n, steps=rng.randint(10, 229), mode=mode)
    if kind == "sir":
        n = _log(rng, 1000, 990_000)
        return dict(kind=kind, n=n, m=rng.randint(2, 4), steps=rng.randint(40, 365),
                    beta=round(rng.uniform(0.01, 0.1), 4), gamma=round(rng.uniform(0.05, 0.2), 4),
                    infected=rng.randint(5, 100), mode=mode)
    if kind == "schelling":
        return dict(kind=kind, h=_log(rng, 24, 640), w=_log(rng, 24, 640),
                    steps=rng.randint(20, 200), mode=mode)
    if kind == "deffuant":
        n, batch = _log(rng, 100, 65_536), _log(rng, 1, 256)
        return dict(kind=kind, n=n, batch=batch, steps=rng.randint(10, 200),
                    ckpt=rng.randint(2, 40), grad=rng.random() < 0.8, mode=mode)
    if kind == "generic":
        return dict(kind=kind, n=_log(rng, 200, 200_000), steps=rng.randint(50, 300))
    return dict(kind=kind, requests=rng.randint(8, 48), n_min=1000,
                n_max=_log(rng, 20_000, 250_000))


# ------------------------------------------------------- what a user has in hand
class _Trader:
    """A generic agent: a position walk with a normal draw and a coin-flip
    wealth change."""

    def init_state(self, cfg, key):
        k1, k2 = jr.split(key)
        return {"x": jr.uniform(k1), "w": jr.randint(k2, (), 0, 6)}

    def update(self, state, model_state, cfg, key):
        k1, k2 = jr.split(key)
        x = jnp.mod(state["x"] + jr.normal(k1) * 0.01, 1.0)
        give = jr.uniform(k2) < 0.5
        return {"x": x, "w": jnp.where(give & (state["w"] > 0), state["w"] - 1, state["w"] + 1)}


def _trader_env(env, agents, params, key):
    new = dict(env)
    new["mean_x"] = jnp.mean(agents["t"]["x"])
    return new


def _trader_metrics(env, agents, params):
    a = agents["t"]
    return {"mean_x": env["mean_x"], "total_w": jnp.sum(a["w"]), "rich": jnp.sum(a["w"] > 3)}


def _deffuant_inputs(case, seed):
    """(eps, mu, target): parameters of every instance, and the statistics of
    a population half settled around two camps."""
    g = np.random.RandomState(seed % (1 << 31))
    eps = g.uniform(0.05, 0.2, case["batch"]).astype(np.float32)
    mu = g.uniform(0.05, 0.3, case["batch"]).astype(np.float32)
    centre = (np.arange(32) + 0.5) / 32
    hist = np.exp(-0.5 * ((centre - 0.3) / 0.06) ** 2) + np.exp(-0.5 * ((centre - 0.75) / 0.09) ** 2)
    target = np.concatenate([[0.5, 0.06], hist / hist.sum()])
    return eps, mu, target


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "seed": int(seed)}
    if kind == "wealth":
        from jaxabm_amd.programs.wealth import WealthEngine

        s["engine"] = WealthEngine(case["n"], seed=seed, mode=case["mode"])
    elif kind == "sir":
        from jaxabm_amd.programs.sir import SIRNetworkEngine

        s["engine"] = SIRNetworkEngine(case["n"], m=case["m"], graph_seed=seed + 1,
                                       beta=case["beta"], gamma=case["gamma"],
                                       n_seed_infected=case["infected"], seed=seed,
                                       mode=case["mode"])
    elif kind == "schelling":
        from jaxabm_amd.programs.schelling import SchellingEngine

        s["engine"] = SchellingEngine(case["h"], case["w"], seed=seed, mode=case["mode"])
    elif kind == "deffuant":
        from jaxabm_amd.programs.deffuant import DeffuantModel

        eps, mu, target = _deffuant_inputs(case, seed)
        s["engine"] = DeffuantModel(case["n"], case["batch"], case["steps"], seed=seed,
                                    ckpt_every=case["ckpt"], mode=case["mode"])
        s["eps"] = torch.from_numpy(eps).to("cuda").requires_grad_(case["grad"])
        s["mu"] = torch.from_numpy(mu).to("cuda").requires_grad_(case["grad"])
        s["target"] = target
    elif kind == "serving":
        from jaxabm_amd.serving import SimulationServer, make_trace, tuned_config

        s["server"] = SimulationServer(tuned_config("batched"))
        s["trace"] = make_trace(case["requests"], seed=seed, n_min=case["n_min"],
                                n_max=case["n_max"])
    return s


# ------------------------------------------------------------------- one pass
def run(state):
    case, seed = state["case"], state["seed"]
    kind = case["kind"]
    if kind == "wealth":
        e = state["engine"]
        e.reset(seed)
        mean, gini = e.run(case["steps"])
        return {"mean": mean, "gini": gini, "x": e.x, "y": e.y, "w": e.w}
    if kind == "sir":
        e = state["engine"]
        e.reset(seed)
        counts = e.run(case["steps"])
        return {"counts": counts, "states": e.states()}
    if kind == "schelling":
        e = state["engine"]
        e.reset(seed)
        happy, moves = e.run(case["steps"])
        return {"happy": happy, "moves": moves, "cells": e.cells, "id": e.id}
    if kind == "deffuant":
        from jaxabm_amd.programs.deffuant import deffuant_loss

        e = state["engine"]
        loss = deffuant_loss(state["eps"], state["mu"], e, state["target"])
        out = {"loss": loss.detach(), "stats": e.stats, "x": e.final_state()}
        if case["grad"]:
            out["eps_grad"], out["mu_grad"] = torch.autograd.grad(
                loss.sum(), (state["eps"], state["mu"]))
        return out
    if kind == "generic":
        with contextlib.redirect_stdout(io.StringIO()):
            m = J.JaxModel(params={}, config=J.ModelConfig(steps=case["steps"], seed=seed),
                           update_state_fn=_trader_env, metrics_fn=_trader_metrics)
            m.add_agent_collection("t", J.AgentCollection(_Trader(), case["n"]))
            hist = m.run(case["steps"], graph=True)
        out = {k: torch.stack(hist[k]) for k in ("mean_x", "total_w", "rich")}
        st = m.agent_collections["t"].states
        return {**out, "x": st["x"], "w": st["w"]}
    server = state["server"]
    tickets = [server.submit(r) for r in state["trace"]]
    server.drain()
    # one row of records per request, as long as the longest request can be
    out = {k: np.zeros((len(tickets), 365), np.float32) for k in ("mean", "gini")}
    out.update({k: np.zeros((len(tickets), 365), np.int32) for k in ("S", "I", "R")})
    for i, t in enumerate(tickets):
        for k, v in server.result(t).items():
            out[k][i, : len(v)] = v
    return out


# ------------------------------------------------------------ what a pass needs
# One threefry block is about 72 integer operations and one normal about 60
# more.  Bytes: state and network once in, state and records once out.
_BLOCK = 72


def _wealth_work(n, steps):
    # per agent-step: an agent key, two walk keys, two normals, two words of
    # the exchange target
    return 12 * n + 8 * steps, n * steps * (7 * _BLOCK + 2 * 60 + 30)


def _sir_work(n, m, steps, gamma):
    # an infected agent draws once a step until it recovers, and each of its
    # edges is drawn at least in its first infected step
    nnz = 2 * m * max(n - m, 1)
    return 4 * (n + 1) + 4 * nnz + n + 12 * steps, _BLOCK * (n / gamma + nnz / 2) * 0.8


def work(case):
    kind = case["kind"]
    if kind == "wealth":
        b, f = _wealth_work(case["n"], case["steps"])
    elif kind == "sir":
        b, f = _sir_work(case["n"], case["m"], case["steps"], case["gamma"])
    elif kind == "schelling":
        # a computed step counts 8 neighbours of every cell; the grid settles
        # after about 30 steps
        nc = case["h"] * case["w"]
        b, f = 5 * nc + 8 * case["steps"], 30 * nc * min(case["steps"], 30)
    elif kind == "deffuant":
        # the initial opinions and the pairings in, the final opinions out;
        # about 40 operations a pair and step forward, 60 in the adjoint
        n, B, S = case["n"], case["batch"], case["steps"]
        b, f = 8 * n * B + 4 * n * S, n // 2 * B * S * (40 + (60 if case["grad"] else 0))
    elif kind == "generic":
        # per agent-step: an agent key, two keys, a normal and a uniform
        n, S = case["n"], case["steps"]
        b, f = 8 * n + 12 * S, n * S * (5 * _BLOCK + 60 + 10)
    else:
        from jaxabm_amd.serving import make_trace

        b = f = 0
        for r in make_trace(case["requests"], seed=0, n_min=case["n_min"], n_max=case["n_max"]):
            rb, rf = (_wealth_work(r.n, r.steps) if r.kind == "wealth"
                      else _sir_work(r.n, r.m, r.steps, r.gamma))
            b, f = b + rb, f + rf
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("sir", "schelling"):
        return "exact"       # counts, and float32 quotients of two counts
    if kind == "deffuant":
        # float32 opinions; the steep gate amplifies their rounding along the
        # run, and the gradients follow it (in long runs without bound: 0.01
        # to 1 against 64 bits at 200 steps)
        return {"rel": 2e-3, "max": 0.05} if case["steps"] <= 60 else {"rel": 0.03, "max": 0.9}
    if kind == "generic":
        # a position within rounding of the modulus wraps a step earlier or
        # later, which the mean of that step shows (measured 1.4e-5)
        return {"rel": 6e-5, "max": 1e-3}
    # float32 positions after up to 229 rounded increments modulo 1 (measured
    # 3.5e-7) and float32 records; whole values (wealth, counts) are exact
    return {"rel": 2e-6, "max": 1e-4}


# ------------------------------------------- the same results in 64 bits (torch)
_M = 0xFFFFFFFF


def _threefry(k0, k1, x0, x1):
    """threefry2x32-20 on Python ints or int64 tensors of 32-bit words."""
    k2 = k0 ^ k1 ^ 0x1BD11BDA
    ks = (k0, k1, k2)
    x0, x1 = (x0 + k0) & _M, (x1 + k1) & _M
    for g in range(5):
        for r in ((13, 15, 26, 6), (17, 29, 16, 24))[g & 1]:
            x0 = (x0 + x1) & _M
            x1 = ((x1 << r) & _M | (x1 >> (32 - r))) ^ x0
        x0 = (x0 + ks[(g + 1) % 3]) & _M
        x1 = (x1 + ks[(g + 2) % 3] + g + 1) & _M
    return x0, x1


def _split2(k, mode):
    """Both halves of split(key); key words are ints or tensors."""
    z = k[0] * 0
    if mode:
        return _threefry(*k, z, z), _threefry(*k, z, z + 1)
    p, q = _threefry(*k, z, z + 2), _threefry(*k, z + 1, z + 3)
    return (p[0], q[0]), (p[1], q[1])


def _scalar_bits(k, mode):
    a, b = _threefry(*k, k[0] * 0, k[0] * 0)
    return a ^ b if mode else a


def _bits(k, n, mode):
    """random.bits(key, (n,)) for a key of ints."""
    e = torch.arange(n, dtype=torch.int64, device="cuda")
    if mode:
        a, b = _threefry(k[0], k[1], e * 0, e)
        return a ^ b
    h = (n + 1) // 2
    lo = e[:h]
    hi = torch.where(h + lo < n, h + lo, lo * 0)
    return torch.cat(_threefry(k[0], k[1], lo, hi))[:n]


def _split(k, n, mode):
    """split(key, n) as a pair of tensors."""
    if mode:
        e = torch.arange(n, dtype=torch.int64, device="cuda")
        return _threefry(k[0], k[1], e * 0, e)
    b = _bits(k, 2 * n, 0)
    return b[0::2], b[1::2]


def _unit(bits):
    return (bits >> 9).double() / float(1 << 23)


def _normal(bits):
    lo = -1.0 + 2.0 ** -24
    u = torch.clamp(_unit(bits) * 2.0 + lo, min=lo)
    return math.sqrt(2.0) * torch.special.erfinv(u)


def _randint(hb, lb, span):
    m = (65536 % span) ** 2 % span
    return (((hb % span) * m + lb % span) & _M) % span


def _step_keys(rng, mode):
    """One step of the model's key schedule: (rng, collection key, env key)."""
    rng, sk = _split2(rng, mode)
    sk, ck = _split2(sk, mode)
    return rng, ck, _split2(sk, mode)[1]


def _wealth_exact(case, seed):
    n, mode = case["n"], case["mode"]
    rng, ik = _split2((seed >> 32 & _M, seed & _M), mode)
    kx, ky = _split2(_split(ik, n, mode), mode)
    x, y = _unit(_scalar_bits(kx, mode)), _unit(_scalar_bits(ky, mode))
    w = torch.ones(n, dtype=torch.int64, device="cuda")
    i = torch.arange(n, dtype=torch.int64, device="cuda")
    wrap = lambda v: (v + (1 << 31)) % (1 << 32) - (1 << 31)  # int32 sums  # noqa: E731
    mean, gini = [], []
    for _ in range(case["steps"]):
        rng, ck, uk = _step_keys(rng, mode)
        k1, k2 = _split2(_split(ck, n, mode), mode)
        x = torch.remainder(x + 0.01 * _normal(_scalar_bits(k1, mode)), 1.0)
        y = torch.remainder(y + 0.01 * _normal(_scalar_bits(k2, mode)), 1.0)
        a, b = _split2(uk, mode)
        t = _randint(_bits(a, n, mode), _bits(b, n, mode), n - 1)
        t = t + (t >= i)
        give = (w > 0).long()
        w = w - give + torch.bincount(t, weights=give.double(), minlength=n).long()
        s, total = int(((i + 1) * torch.sort(w)[0]).sum()), int(w.sum())
        mean.append(total / n)
        gini.append(wrap(2 * s) / wrap(n * total) - (n + 1) / n if total > 1e-6 else 0.0)
    return {"mean": np.array(mean), "gini": np.array(gini), "x": x, "y": y, "w": None}


def _generic_exact(case, seed):
    n = case["n"]
    rng, ik = _split2((seed >> 32 & _M, seed & _M), 1)
    k1, k2 = _split2(_split(ik, n, 1), 1)
    x = _unit(_scalar_bits(k1, 1))
    a, b = _split2(k2, 1)
    w = _randint(_scalar_bits(a, 1), _scalar_bits(b, 1), 6)
    mean = []
    for _ in range(case["steps"]):
        rng, ck, _uk = _step_keys(rng, 1)
        k1, k2 = _split2(_split(ck, n, 1), 1)
        x = torch.remainder(x + 0.01 * _normal(_scalar_bits(k1, 1)), 1.0)
        give = (_unit(_scalar_bits(k2, 1)) < 0.5) & (w > 0)
        w = torch.where(give, w - 1, w + 1)
        mean.append(float(x.mean()))
    return {"mean_x": np.array(mean), "total_w": None, "rich": None, "x": x, "w": None}


def _permutation(k, n, mode):
    p = torch.arange(n, dtype=torch.int64, device="cuda")
    for _ in range(math.ceil(3.0 * math.log(max(1, n)) / math.log(4294967295.0))):
        k, sub = _split2(k, mode)
        p = p[torch.sort(_bits(sub, n, mode), stable=True)[1]]
    return p


def _deffuant_exact(case, seed):
    n, B, mode = case["n"], case["batch"], case["mode"]
    eps, mu, target = _deffuant_inputs(case, seed)
    eps = torch.from_numpy(eps).cuda().double()
    mu = torch.from_numpy(mu).cuda().double()
    target = torch.from_numpy(target).cuda()
    rng, ik = _split2((seed >> 32 & _M, seed & _M), mode)
    x = _unit(_scalar_bits(_split(ik, n, mode), mode))[:, None].repeat(1, B)
    tape = []
    for _ in range(case["steps"]):
        rng, _ck, uk = _step_keys(rng, mode)
        p = _permutation(uk, n, mode)
        a, c = p[0: n // 2 * 2: 2], p[1::2]
        d = x[c] - x[a]
        delta = mu * torch.sigmoid((eps - d.abs()) / 0.02) * d
        x[a] += delta
        x[c] -= delta
        tape.append((a, c, d))
    xf = x.detach().requires_grad_(True)
    stats = [xf.mean(0), xf.var(0, unbiased=False)]
    prev = torch.sigmoid(128.0 * xf).mean(0)
    for k in range(1, 33):
        cur = torch.sigmoid(128.0 * (xf - k / 32.0)).mean(0)
        stats.append(prev - cur)
        prev = cur
    stats = torch.stack(stats, 1)
    loss = ((stats - target) ** 2).sum(1)
    out = {"loss": loss.detach(), "stats": stats.detach(), "x": x}
    if case["grad"] and case["steps"] > 60:
        # a float32 run's gradient is that of its own rounded trajectory
        out["eps_grad"] = out["mu_grad"] = None
    elif case["grad"]:
        lam, = torch.autograd.grad(loss.sum(), xf)
        ge, gm = torch.zeros_like(eps), torch.zeros_like(mu)
        for a, c, d in reversed(tape):
            g = torch.sigmoid((eps - d.abs()) / 0.02)
            gp = g * (1 - g) / 0.02
            v = lam[a] - lam[c]
            ge += (v * (mu * d * gp)).sum(0)
            gm += (v * (g * d)).sum(0)
            fd = v * (mu * (g - d.abs() * gp))
            lam[a] -= fd
            lam[c] += fd
        out["eps_grad"], out["mu_grad"] = ge, gm
    return out


def exact(case, seed):
    # SIR, Schelling: whole numbers and quotients of two of them.  Serving:
    # dozens of simulations, far beyond 20 seconds this way.
    fn = {"wealth": _wealth_exact, "generic": _generic_exact,
          "deffuant": _deffuant_exact}.get(case["kind"])
    return fn(case, int(seed)) if fn else None
