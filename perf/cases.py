"""Timed cases: the work a user of piqmc has the framework do.

Every case is one pass through a public entry point (``piqmc.device``,
``piqmc.pipeline``, ``piqmc.qmc``, ``piqmc.made``) on inputs made from a seed.
A case is a dict of plain values; ``kind`` names the entry point:

  qa        Problem.qa_colored, the parallel sweep (lattice or SK couplings)
  pipeline  pipeline.anneal: preanneal, tile, quantum anneal, slice energies
  batch     device.Batch: a heterogeneous mix in one persistent launch
  replay    Problem.qa_replay, the bit-exact replay of R replicas
  dropin    qmc.QuantumAnneal on host arrays, the reference's own call
  fit       made.MADE.fit, one epoch of training
  learned   made.anneal_with_proposals, the sweep with network moves

Couplings (``model``): ``pm`` +-1 bonds, ``pmh`` +-1 bonds with Gaussian
fields of width 0.1, ``gauss`` N(0,1) bonds, ``uniform`` U[-2,2] bonds (what the
reference's generator draws), ``sk`` dense N(0,1/N).
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "pathintegral-qmc_amd"))

GAMMA0, GAMMA1 = 3.0, 1e-8   # transverse field, start and end of every schedule


def _qa(model, L, dim, P, R, S, M=1, T=None, trace=False):
    return {"kind": "qa", "model": model, "L": L, "dim": dim, "P": P, "R": R, "S": S, "M": M,
            "T": 1.0 / P if T is None else T, "trace": trace}


def listed():
    return [
        # The smallest call: one replica of the 64-spin glass, where launches,
        # allocations and uploads are all there is.
        dict(_qa("pm", 8, 2, 20, 1, 100), name="pm 8x8 one replica"),
        # The headline: 4096 replicas of the 1024-spin +-J glass.
        dict(_qa("pm", 32, 2, 64, 4096, 500), name="pm 32x32 headline"),
        # An odd lattice (no two-coloring), ragged slices and replicas, several
        # sweeps per field and the energy trace a user plots.
        dict(_qa("pm", 33, 2, 50, 301, 60, M=2, trace=True), name="pm 33x33 ragged trace"),
        # +-1 bonds with fields on the cubic lattice, 128 slices.
        dict(_qa("pmh", 12, 3, 128, 1024, 100), name="pm fields 12^3"),
        # The reference's example run (preanneal 3 -> 0.01, tile over P=20
        # slices, anneal at T=0.01, energy of every slice) at the size of its
        # 80x80 instance with Gaussian bonds.
        {"kind": "pipeline", "name": "gauss 80x80 pipeline", "model": "gauss", "L": 80, "dim": 2,
         "P": 20, "R": 32, "S": 40, "T": 0.01},
        # The three-dimensional Edwards-Anderson glass, with its energy trace.
        dict(_qa("gauss", 10, 3, 64, 128, 30, trace=True), name="gauss 10^3 trace"),
        # A dense Sherrington-Kirkpatrick glass, few replicas.
        dict(_qa("sk", 256, 1, 32, 16, 50), name="sk 256"),
        # Many instances of several sizes in one persistent launch.
        {"kind": "batch", "name": "batch of 48", "jobs": 48, "reps": 2, "smax": 200, "mix": 0},
        # Bit-exact replay of many replicas of the 1024-spin glass.
        {"kind": "replay", "name": "replay 32x32", "model": "pm", "L": 32, "dim": 2, "P": 64, "R": 2048,
         "S": 5, "M": 1, "T": 1.0 / 64},
        # The reference's call on host arrays: the 64-spin workload.
        {"kind": "dropin", "name": "QuantumAnneal 8x8", "model": "pm", "L": 8, "dim": 2, "P": 20, "S": 100,
         "M": 1, "T": 0.05},
        # One epoch of the 256-spin proposal network.
        {"kind": "fit", "name": "fit 256-512", "N": 256, "H": 512, "rows": 8192, "batch": 1024},
        # A sweep of the 256-spin glass with a network move every four steps.
        {"kind": "learned", "name": "learned 16x16", "L": 16, "P": 32, "R": 2048, "S": 20, "every": 4, "H": 512},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _even(rng, lo, hi):
    return max(lo, _log(rng, lo, hi) // 2 * 2)


def draw(rng):
    kind = rng.choice(["qa", "qa", "qa", "qa", "pipeline", "batch", "replay", "dropin", "fit", "learned"])
    if kind == "qa":
        model = rng.choice(["pm", "pm", "pmh", "gauss", "uniform", "sk"])
        dim = 1 if model == "sk" else rng.choice([2, 3])
        L = {1: _log(rng, 40, 256), 2: _log(rng, 6, 80), 3: _log(rng, 4, 12)}[dim]
        P = _even(rng, 8, 128)
        N = L ** dim
        # spin words a sweep updates (both parities), up to what the listed
        # cases of the same couplings take
        cap = {"pm": 5e8, "pmh": 1.5e8, "gauss": 1.2e7, "uniform": 1.2e7, "sk": 2e5}[model]
        R = min(_log(rng, 1, 2048 if model != "sk" else 64), max(1, int(cap / (20.0 * N))))
        S = max(5, min(_log(rng, 10, 500), int(cap / (2.0 * N * R))))
        return _qa(model, L, dim, P, R, S, T=rng.choice([0.01, 1.0 / P, 2.0 / P]), trace=rng.random() < 0.3)
    if kind == "pipeline":
        L = _log(rng, 8, 80)
        R = min(_log(rng, 1, 128), int(8e4 / (L * L)) + 1)
        return {"kind": kind, "model": rng.choice(["uniform", "gauss", "pm"]), "L": L, "dim": 2,
                "P": _even(rng, 8, 40), "R": R, "S": _log(rng, 10, 40), "T": 0.01}
    if kind == "batch":
        return {"kind": kind, "jobs": _log(rng, 6, 48), "reps": rng.choice([1, 2, 3]),
                "smax": _log(rng, 110, 200), "mix": rng.randrange(1, 1000)}
    if kind == "replay":
        L = _log(rng, 8, 40)
        P = _log(rng, 4, 64)
        R = _log(rng, 64, 2048)
        S = max(1, min(40, int(3e8 / (L * L * P * R))))
        return {"kind": kind, "model": rng.choice(["pm", "gauss"]), "L": L, "dim": 2, "P": P, "R": R, "S": S,
                "M": 1, "T": 1.0 / P}
    if kind == "dropin":
        L = _log(rng, 4, 16)
        P = _log(rng, 4, 30)
        S = max(4, min(_log(rng, 20, 100), int(128000 / (L * L * P))))
        return {"kind": kind, "model": rng.choice(["pm", "gauss"]), "L": L, "dim": 2, "P": P, "S": S, "M": 1,
                "T": rng.choice([0.05, 0.2])}
    N = rng.choice([36, 64, 100, 121, 225, 256])
    H = 64 * rng.randint(1, 8)
    if kind == "fit":
        batch = rng.choice([256, 500, 1024])
        return {"kind": kind, "N": N, "H": H, "rows": batch * rng.randint(2, 8) + rng.randint(0, 99),
                "batch": batch}
    return {"kind": "learned", "L": rng.choice([8, 11, 16]), "P": _even(rng, 8, 32), "R": _log(rng, 64, 2048),
            "S": rng.randint(8, 24), "every": rng.choice([2, 4]), "H": 64 * rng.randint(1, 3)}


# ------------------------------------------------------------------ inputs
def _instance(model, L, dim, rs):
    """(N, neighbour table) of an instance with couplings drawn from rs."""
    from piqmc import instances
    if model == "sk":
        N, r, c, v = instances.sk(L, rs)
    else:
        N, r, c, v = instances.lattice_pm_j(L, dim, rs, 0.1 if model == "pmh" else 0.0)
        if model == "gauss":
            v = rs.normal(0.0, 1.0, v.size)
        elif model == "uniform":
            v = rs.uniform(-2.0, 2.0, v.size)
    return N, instances.neighbors(N, r, c, v)


def _spins(shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(0, 2, shape, generator=g, dtype=torch.int8, device="cuda") * 2 - 1


def prepare(case, seed):
    from piqmc import device, made, workloads
    k = case["kind"]
    rs = np.random.RandomState(seed & 0x7FFFFFFF)
    if k in ("qa", "pipeline", "replay", "dropin"):
        N, nbs = _instance(case["model"], case["L"], case["dim"], rs)
    st = {"case": case, "seed": seed}
    if k == "qa":
        st.update(pb=device.Problem(nbs), sched=np.linspace(GAMMA0, GAMMA1, case["S"]),
                  init=_spins((case["R"], case["P"], N), seed))
        st["confs"] = torch.empty_like(st["init"])
    elif k == "pipeline":
        st.update(pb=device.Problem(nbs), init=_spins((case["R"], N), seed),
                  pre=np.linspace(3.0, 0.01, case["S"]), field=np.linspace(1.5, GAMMA1, case["S"]))
    elif k == "batch":
        probs, st["jobs"] = {}, []
        for j in workloads.batch_mix(case["jobs"], case["reps"], seed=case["mix"]):
            key = j["kind"], j["size"]
            if key not in probs:
                j2 = dict(j, iseed=j["iseed"] + seed % 100003)
                probs[key] = device.Problem(workloads.batch_instance(j2)[1])
            S = max(2, j["S"] * case["smax"] // 1000)
            init = _spins((case["reps"], j["P"], probs[key].nspins), seed + j["t"])
            st["jobs"].append((probs[key], init, np.linspace(GAMMA0, GAMMA1, S), j))
    elif k == "replay":
        R, G = case["R"], case["S"] * case["M"]
        seeds = rs.randint(0, 2**31 - 1, R).astype(np.uint32)
        st.update(pb=device.Problem(nbs), sched=np.linspace(GAMMA0, GAMMA1, case["S"]),
                  init=_spins((R, case["P"], N), seed),
                  perms=torch.from_numpy(device.perm_streams(seeds, N, G).view(np.int16)).cuda(),
                  rand=torch.from_numpy(device.rand_states(seeds).view(np.int32)).cuda())
    elif k == "dropin":
        st.update(nbs=nbs, N=N, sched=np.linspace(GAMMA0, GAMMA1, case["S"]),
                  init=np.asfortranarray(rs.randint(0, 2, (N, case["P"])) * 2.0 - 1.0))
    elif k == "fit":
        st.update(net=made.MADE(case["N"], case["H"], case["H"], seed=seed & 0xFFFFFF),
                  data=torch.from_numpy(_rows(case, seed)).cuda())
    else:
        N, nbs = _instance("pm", case["L"], 2, rs)
        st.update(pb=device.Problem(nbs), net=made.MADE(N, case["H"], case["H"], seed=seed & 0xFFFFFF),
                  init=_spins((case["R"], case["P"], N), seed), sched=np.linspace(1.0, GAMMA1, case["S"]))
    return st


def _rows(case, seed):
    """Training slices: chains of correlated spins, as an annealed slice has."""
    rs = np.random.RandomState(seed & 0x7FFFFFFF)
    keep = rs.rand(case["rows"], case["N"]) < 0.8
    keep[:, 0] = rs.rand(case["rows"]) < 0.5
    return np.ascontiguousarray(np.cumprod(np.where(keep, 1, -1), axis=1).astype(np.int8))


# ------------------------------------------------------------------ one pass
def run(state):
    from piqmc import device, made, pipeline, qmc
    case, seed = state["case"], state["seed"]
    k = case["kind"]
    if k == "qa":
        confs = state["confs"]
        confs.copy_(state["init"])
        et = state["pb"].qa_colored(confs, state["sched"], case["M"], case["T"], seed, trace=case["trace"])
        return {"confs": confs, "trace": et}
    if k == "pipeline":
        r = pipeline.anneal(state["pb"], case["R"], case["P"], case["T"], state["field"], pre_sched=state["pre"],
                            seed=seed, init=state["init"].clone())
        return {"confs": r.confs, "energies": r.energies, "best_energy": r.best_energy, "best_conf": r.best_conf}
    if k == "batch":
        b, outs = device.Batch(), []
        for pb, init, sched, j in state["jobs"]:
            outs.append(init.clone())
            b.add(pb, outs[-1], sched, 1, j["T"], j["seed"] + seed, j["replica_base"])
        b.run()
        return {"confs": outs}
    if k == "replay":
        confs, rand = state["init"].clone(), state["rand"].clone()
        draws, ties = state["pb"].qa_replay(confs, state["sched"], case["M"], case["T"], state["perms"], rand)
        return {"confs": confs, "rand": rand, "draws": draws, "ties": ties}
    if k == "dropin":
        confs = state["init"].copy(order="F")
        rng = np.random.RandomState(seed & 0x7FFFFFFF)
        ctypes.CDLL(None).srand(seed & 0x7FFFFFFF)
        qmc.QuantumAnneal(state["sched"], case["M"], case["P"], case["T"], state["N"], confs, state["nbs"], rng)
        return {"confs": confs}
    if k == "fit":
        nll = state["net"].fit(state["data"], epochs=1, batch=case["batch"], lr=1e-3, seed=seed & 0xFFFF)
        return {"nll": nll, "params": state["net"].params()}
    confs = state["init"].clone()
    made.anneal_with_proposals(state["pb"], state["net"], confs, state["sched"], 1, 1.0 / case["P"], seed,
                               every=case["every"])
    return {"confs": confs}


# ------------------------------------------------------------------ work
def _degree(case):
    if case["model"] == "sk":
        return case["L"] - 1
    return 2 * case["dim"] + (1 if case["model"] == "pmh" else 0)


def work(case):
    """An attempt cannot do without its row's terms, the two Trotter terms and
    the comparison; the state is read and written once, a table entry (index
    and coupling, 8 bytes) read once."""
    k = case["kind"]
    if k in ("qa", "pipeline", "replay", "dropin"):
        N = case["L"] ** case["dim"]
        z, R, M = _degree(case), case.get("R", 1), case.get("M", 1)
        flops = (z + 3.0) * N * case["P"] * R * case["S"] * M
        nbytes = 2.0 * R * case["P"] * N + 8.0 * N * z + 8.0 * case["S"]
        if k == "pipeline":
            flops += (z + 1.0) * N * R * case["S"] + (z + 1.0) * N * R * case["P"]
            nbytes += 2.0 * R * N + 8.0 * R * case["P"]
        if k == "replay":
            nbytes += 2.0 * case["S"] * M * N * R + 256.0 * R
        if k == "dropin":
            nbytes += 14.0 * R * case["P"] * N
        return {"bytes": nbytes, "flops": flops}
    if k == "batch":
        from piqmc import workloads
        nbytes = flops = 0.0
        for j in workloads.batch_mix(case["jobs"], case["reps"], seed=case["mix"]):
            sk = j["kind"] == "sk"
            N, z = (j["size"], j["size"] - 1) if sk else (j["size"] ** 2, 4)
            S = max(2, j["S"] * case["smax"] // 1000)
            nbytes += 2.0 * case["reps"] * j["P"] * N + 8.0 * N * z + 8.0 * S
            flops += (z + 3.0) * N * j["P"] * case["reps"] * S
        return {"bytes": nbytes, "flops": flops}
    if k == "fit":
        N, H, steps = case["N"], case["H"], case["rows"] // case["batch"]
        params = 2.0 * N * H + H * H
        return {"bytes": 1.0 * case["rows"] * N + 24.0 * params, "flops": 6.0 * params * steps * case["batch"]}
    N, rounds = case["L"] ** 2, -(-case["S"] // case["every"])
    params = 2.0 * N * case["H"] + case["H"] ** 2
    return {"bytes": 2.0 * case["R"] * case["P"] * N + 2.0 * params,
            "flops": 7.0 * N * case["P"] * case["R"] * case["S"] + rounds * 2.0 * case["R"] * 2.0 * params}


# ------------------------------------------------------------------ 64 bits
def _made_init(N, H, seed):
    """The network's initial float32 weights and its masks: U(-1, 1)/sqrt(fan
    in) from a 64-bit linear congruential generator, drawn in row order for
    the unmasked entries."""
    a, c, m64 = 6364136223846793005, 1442695040888963407, (1 << 64) - 1
    deg = 1 + np.arange(H) % (N - 1)
    d = np.arange(N)
    masks = [deg[:, None] >= d[None, :] + 1, deg[:, None] >= deg[None, :], d[:, None] + 1 > deg[None, :]]
    x, ws = (seed * a + c) & m64, []
    for mk in masks:
        n, vals = int(mk.sum()), []
        for _ in range(n):
            x = (x * a + c) & m64
            vals.append(x >> 11)
        w = np.zeros(mk.shape, np.float32)
        w[mk] = ((np.array(vals, np.float64) / 2.0**53 * 2.0 - 1.0) / math.sqrt(mk.shape[1])).astype(np.float32)
        ws.append(w)
    return ws, masks


def exact(case, seed):
    """The epoch of training in float64: the mean loss.  (Adam divides every
    gradient by its own size, so the weights of parameters whose gradient is
    rounding noise have no value in 64 bits to be compared with.)  The other
    kinds return spins, and energies of those very spins."""
    if case["kind"] != "fit":
        return None
    ws, masks = _made_init(case["N"], case["H"], seed & 0xFFFFFF)
    W = [torch.from_numpy(w.astype(np.float64)) for w in ws]
    Mk = [torch.from_numpy(m.astype(np.float64)) for m in masks]
    b = [torch.zeros(w.shape[0], dtype=torch.float64) for w in ws]
    p = [W[0], b[0], W[1], b[1], W[2], b[2]]
    data = torch.from_numpy(_rows(case, seed).astype(np.float64))
    g = torch.Generator(device="cpu").manual_seed(seed & 0xFFFF)
    perm = torch.randperm(case["rows"], generator=g)
    m1 = [torch.zeros_like(t) for t in p]
    m2 = [torch.zeros_like(t) for t in p]
    steps, total = case["rows"] // case["batch"], 0.0
    for t in range(steps):
        x = data[perm[t * case["batch"]:(t + 1) * case["batch"]]]
        q = [v.clone().requires_grad_(True) for v in p]
        h = torch.relu(x @ (q[0] * Mk[0]).T + q[1])
        h = torch.relu(h @ (q[2] * Mk[1]).T + q[3])
        lo = h @ (q[4] * Mk[2]).T + q[5]
        loss = (torch.nn.functional.softplus(lo) - lo * (x < 0)).sum(1).mean()
        loss.backward()
        total += float(loss.detach())
        for i in range(6):
            gr = q[i].grad
            m1[i] = 0.9 * m1[i] + 0.1 * gr
            m2[i] = 0.999 * m2[i] + 0.001 * gr * gr
            c1, c2 = 1 - 0.9 ** (t + 1), 1 - 0.999 ** (t + 1)
            p[i] = p[i] - 1e-3 * (m1[i] / c1) / (torch.sqrt(m2[i] / c2) + 1e-8)
    return {"nll": [total / steps], "params": [None] * 6}
