"""The framework's own performance cases: what a program that uses it has it do.

Each case is one call (or one fixed sequence of calls) through the Python binding of the C
ABI, on inputs made from a seed. The sizes are those of this repository's configurations,
tests and benchmark: the 306,328-bit muon QUBO and the range of the serving stream (2k to
300k voxels, 1k to 75k rays, 8 to 16 branches), the gravimetry QUBO, the N = 800 max-cut, the
batched sparse QUBOs, the dense precision study, the exact region posterior, and the
reference's own trajectories.

  listed()             the cases
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  the inputs and handles a program holds before the call
  run(state)           one pass; returns its outputs
  work(case)           the bytes and flops one pass cannot do without
  exact(case, seed)    the outputs in 64 bits from plain torch or numpy, where there are any
"""
import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

import qublar_amd as qa


def muon_case(grid, th, branches, precision, recompute, anneal, hold, keep):
    """A muon request: a pyramid of grid^3 voxels (about 0.146 grid^3 bits) seen from three
    chambers through min(360, 5 th) x th sky bins each."""
    return dict(kind="muon", grid=grid, th=th, branches=branches, precision=precision, recompute=recompute,
                anneal=anneal, hold=hold, keep=keep)


def listed():
    return [
        # The headline solve: the whole pyramid, 16 branches annealed to T = 1 with FP32
        # residuals; the caller takes the agreement maps and energies.
        dict(muon_case(128, 70, 16, "fp32", 50, 200, 50, False), name="muon_full_fp32"),
        # A small request of the serving stream (about 2k voxels), answered alone: the latency
        # a lightly loaded server shows.
        dict(muon_case(24, 8, 8, "fp32", 10, 200, 50, True), name="muon_request_small"),
        # A request from the middle of the stream's range in the reference's arithmetic (FP64
        # residuals), as a user does who wants its answer without a carry error.
        dict(muon_case(55, 24, 16, "fp64", 0, 200, 50, True), name="muon_request_mid_fp64"),
        # The gravimetry QUBO (200 stations per cell, thousands of colour classes): the first
        # sweeps of its anneal, FP64 residuals.
        dict(kind="gravity", nx=100, ny=200, nz=10, h=5.0, radius=50.0, branches=16, precision="fp64", recompute=0,
             anneal=8, hold=2, name="gravity_fp64"),
        # The evidence of finished branches: FP64 energies of 16 states of the full muon QUBO,
        # data and prior apart.
        dict(kind="energy", grid=128, th=70, states=16, name="muon_evidence"),
        # The plain max-cut workload: 16 replicas of an N = 800 graph, 1000 sweeps.
        dict(kind="maxcut", n=800, degree=48.0, signed=True, replicas=16, anneal=1000, hold=0, t_hot=3.0, t_cold=0.05,
             reference=False, name="maxcut_16"),
        # The reference's GPU benchmark shape (G1-like graph, unit weights, scaled budget) with
        # many replicas: throughput.
        dict(kind="maxcut", n=800, degree=48.0, signed=False, replicas=8192, anneal=950, hold=50, t_hot=0.0,
             t_cold=0.1, reference=False, name="maxcut_batch"),
        # The same engine in the reference's own trajectory, which the drop-in run_batch gives.
        dict(kind="maxcut", n=800, degree=48.0, signed=False, replicas=2048, anneal=950, hold=50, t_hot=0.0,
             t_cold=0.1, reference=True, name="maxcut_reference"),
        # branch_fractions in the reference's own trajectory: many branches of a small request.
        dict(kind="muon_reference", grid=32, th=20, branches=1024, anneal=40, hold=10, name="muon_reference"),
        # Many uneven sparse QUBOs in one persistent launch, the launch shape tuned once.
        dict(kind="qubo", instances=48, n_lo=1000, n_hi=16384, degrees="3,8,32,64", r_lo=8, r_hi=32, sweeps=400,
             name="qubo_batch"),
        # A dense QUBO with FP32 fields and the FP64 recompute every 10 sweeps.
        dict(kind="dense", n=2048, replicas=32, precision="fp32", recompute=10, sweeps=400, name="dense_fp32"),
        # The exact posterior of a region of 26 bits.
        dict(kind="roi", n=26, beta=1.0, name="roi_26"),
    ]


def log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def muon_size(voxels, rays):
    """The serving stream's scene for about `voxels` bits and `rays` rays."""
    grid = min(128, max(24, round((voxels / 0.146) ** (1.0 / 3.0))))
    return grid, min(70, max(4, round(math.sqrt(rays / 15.0))))


def draw(rng):
    kind = rng.choice(["muon", "muon", "muon", "gravity", "energy", "maxcut", "maxcut", "muon_reference", "qubo",
                       "dense", "roi"])
    if kind == "muon":
        grid, th = muon_size(math.exp(rng.uniform(math.log(2e3), math.log(2.4e5))),
                             math.exp(rng.uniform(math.log(1e3), math.log(6e4))))
        fp32 = rng.random() < 0.6
        return muon_case(grid, th, rng.randint(8, 16), "fp32" if fp32 else "fp64",
                         rng.choice([10, 25, 50]) if fp32 else 0, rng.randint(40, 160), rng.randint(0, 40),
                         rng.random() < 0.5)
    if kind == "gravity":
        fp32 = rng.random() < 0.5
        return dict(kind="gravity", nx=log_int(rng, 20, 80), ny=log_int(rng, 20, 120), nz=rng.randint(4, 10),
                    h=5.0, radius=rng.choice([20.0, 30.0, 50.0]), branches=rng.randint(4, 16),
                    precision="fp32" if fp32 else "fp64", recompute=5 if fp32 else 0, anneal=8, hold=2)
    if kind == "energy":
        grid, th = muon_size(math.exp(rng.uniform(math.log(2e3), math.log(3e5))),
                             math.exp(rng.uniform(math.log(1e3), math.log(7.5e4))))
        return dict(kind="energy", grid=grid, th=th, states=rng.randint(1, 16))
    if kind == "maxcut":
        n = log_int(rng, 100, 2000)
        anneal = log_int(rng, 50, 1000)
        most = min(8192.0, 3.0e9 / (n * (anneal + 20)))   # below the listed batch's 6.6e9 updates
        reference = rng.random() < 0.4
        return dict(kind="maxcut", n=n, degree=min(n / 4.0, rng.uniform(4.0, 48.0)), signed=rng.random() < 0.5,
                    replicas=log_int(rng, 1, most / 4.0 if reference else most), anneal=anneal,
                    hold=rng.randint(0, 20), t_hot=0.0, t_cold=0.1, reference=reference)
    if kind == "muon_reference":
        return dict(kind="muon_reference", grid=rng.randint(24, 32), th=rng.randint(8, 20),
                    branches=log_int(rng, 16, 1024), anneal=rng.randint(10, 36), hold=rng.randint(0, 8))
    if kind == "qubo":
        return dict(kind="qubo", instances=log_int(rng, 4, 40), n_lo=1000, n_hi=log_int(rng, 2000, 16384),
                    degrees=rng.choice(["3,8,32,64", "3,8", "8,32", "64"]), r_lo=rng.randint(1, 8),
                    r_hi=rng.randint(8, 32), sweeps=rng.randint(50, 300))
    if kind == "dense":
        fp32 = rng.random() < 0.6
        return dict(kind="dense", n=log_int(rng, 100, 2048), replicas=log_int(rng, 1, 96),
                    precision="fp32" if fp32 else "fp64", recompute=rng.choice([1, 10, 100]) if fp32 else 0,
                    sweeps=rng.randint(50, 250))
    return dict(kind="roi", n=rng.randint(8, 30), beta=rng.choice([0.5, 1.0, 2.0]))


# ---- inputs -----------------------------------------------------------------------------

PRECISION = {"fp64": qa.FP64, "fp32": qa.FP32}


def muon_arrays(case, seed):
    th = case["th"]
    return qa.muon_scene(grid=case["grid"], sky_az=min(360, 5 * th), sky_th=th,
                         log2_muons=27 if case["grid"] == 128 else 24, seed=1000 + seed)


def branch_like_states(P, states, seed):
    """Finished branches as they look: the void found, 1% of the voxels off."""
    rng = np.random.default_rng([seed, 5])
    return (P.truth[None, :] ^ (rng.random((states, P.n_vars)) < 0.01)).astype(np.uint8)


def maxcut_graph(case, seed):
    g = qa.er_graph(case["n"], min(1.0, case["degree"] / max(1, case["n"] - 1)), 1 + seed)
    return g if case["signed"] else qa.GraphArrays(g.n, g.eu, g.ev, np.abs(g.ew))


def region(case, seed):
    """A region's conditional QUBO: h ~ N(0, 2), J_ij ~ N(0, 1) above the diagonal."""
    rng = np.random.default_rng([seed, 31])
    n = case["n"]
    return rng.normal(0, 2, n), np.triu(rng.normal(0, 1, (n, n)), 1)


def qubo_instances(case, seed):
    """The batch of qa.qubo_batch_workload with sizes, degrees and replicas that the case alone
    fixes (n log-uniform); graphs, couplings and draws are the seed's."""
    shape, rng = np.random.default_rng(2026), np.random.default_rng([seed, 7])
    degrees = [int(d) for d in case["degrees"].split(",")]
    specs = []
    for _ in range(case["instances"]):
        n = int(np.exp(shape.uniform(np.log(case["n_lo"]), np.log(case["n_hi"]))))
        specs.append((n, int(shape.choice(degrees)), int(rng.integers(1, 2**62)),
                      int(shape.integers(case["r_lo"], case["r_hi"] + 1))))
    with ThreadPoolExecutor(8) as ex:
        return list(ex.map(lambda s: qa.random_regular_qubo(*s), specs))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "muon":
        return dict(kind=kind, problem=qa.Problem(muon_arrays(case, seed)),
                    sched=qa.schedule(50.0, 1.0, case["anneal"], case["hold"]), branches=case["branches"],
                    precision=PRECISION[case["precision"]], recompute=case["recompute"], keep=case["keep"], seed=seed)
    if kind == "gravity":
        hx, hy, hz = 0.5 * case["nx"] * case["h"], 0.5 * case["ny"] * case["h"], 0.3 * case["nz"] * case["h"]
        body = dict(body_lo=(0.8 * hx, 0.8 * hy, -2.0 * hz), body_hi=(1.2 * hx, 1.2 * hy, -hz))
        P = qa.gravity_scene(nx=case["nx"], ny=case["ny"], nz=case["nz"], h=case["h"], radius=case["radius"],
                             seed=1000 + seed, **body)
        return dict(kind="muon", problem=qa.Problem(P),
                    sched=qa.schedule(50.0, 1.0, case["anneal"], case["hold"]), branches=case["branches"],
                    precision=PRECISION[case["precision"]], recompute=case["recompute"], keep=True, seed=seed)
    if kind == "energy":
        P = muon_arrays(case, seed)
        return dict(kind=kind, problem=qa.Problem(P), X=branch_like_states(P, case["states"], seed))
    if kind == "maxcut":
        g = maxcut_graph(case, seed)
        t_hot = case["t_hot"] or float(np.sqrt(2.0 * np.sum(g.ew.astype(np.float64) ** 2) / g.n)) or 1.0
        return dict(kind=kind, graph=qa.Graph(g), sched=qa.schedule(t_hot, case["t_cold"], case["anneal"], case["hold"]),
                    replicas=case["replicas"], reference=case["reference"], seed=1 + seed)
    if kind == "muon_reference":
        return dict(kind=kind, problem=qa.Problem(muon_arrays(case, seed)),
                    sched=qa.schedule(50.0, 1.0, case["anneal"], case["hold"]), branches=case["branches"], seed=seed)
    if kind == "qubo":
        batch = qa.QuboBatch(qubo_instances(case, seed))
        # the launch shape is tuned once per batch, as a program does that anneals it more than once
        rep = batch.anneal(qa.schedule(5.0, 0.05, 8, 0), x=False, energy=False)["report"]
        return dict(kind=kind, batch=batch, sched=qa.schedule(5.0, 0.05, case["sweeps"], 0),
                    replica_block=rep["replica_block"], block=rep["block"])
    if kind == "dense":
        Q, h = qa.dense_qubo(case["n"], 4096 + seed)
        return dict(kind=kind, dense=qa.DenseQubo(Q, h), sched=qa.schedule(1.0, 0.01, case["sweeps"], 0),
                    replicas=case["replicas"], precision=PRECISION[case["precision"]], recompute=case["recompute"],
                    seed=seed)
    h, J = region(case, seed)
    return dict(kind="roi", h=h, J=J, beta=case["beta"])


def run(state):
    kind = state["kind"]
    if kind == "muon":
        out = state["problem"].anneal_branches(state["sched"], state["branches"], state["seed"], state["precision"],
                                               state["recompute"], branches=state["keep"])
        return {k: out[k] for k in ("branches", "p_void", "tri", "certainty", "energy") if out[k] is not None}
    if kind == "energy":
        total, data, prior = state["problem"].energy(state["X"])
        return dict(total=total, data=data, prior=prior)
    if kind == "maxcut":
        anneal = state["graph"].run_batch_reference if state["reference"] else state["graph"].run_batch
        spins, energy, _ = anneal(state["sched"], state["seed"], state["replicas"])
        return dict(spins=spins, energy=energy)
    if kind == "muon_reference":
        out = state["problem"].anneal_branches_reference(state["sched"], state["branches"], state["seed"],
                                                         branches=False)
        return {k: out[k] for k in ("p_void", "tri", "certainty", "energy")}
    if kind == "qubo":
        out = state["batch"].anneal(state["sched"], replica_block=state["replica_block"], block=state["block"])
        return dict(x=np.concatenate([x.reshape(-1) for x in out["x"]]), energy=np.concatenate(out["energy"]))
    if kind == "dense":
        out = state["dense"].anneal(state["sched"], state["replicas"], state["seed"], state["precision"],
                                    state["recompute"])
        return dict(x=out["x"], energy=out["energy"])
    out = qa.roi_enumerate(state["h"], state["J"], state["beta"])
    return {k: out[k] for k in ("marginal", "map_state", "e_min", "log_z", "p_map")}


# ---- what a pass cannot do without --------------------------------------------------------

def muon_work(case):
    """Bits, rays and entries of a muon scene, from the full one's 306,328 / 75,600 / 3,829,376:
    a ray crosses voxels in proportion to the grid's edge."""
    n = 306328.0 * (case["grid"] / 128.0) ** 3
    rays = 3.0 * min(360, 5 * case["th"]) * case["th"]
    return n, rays, 50.65 * rays * case["grid"] / 128.0


def gravity_work(case):
    """Cells, stations and entries: a cell at depth z sees the stations within
    sqrt(radius^2 - z^2) of its column."""
    n, rays, h, r = case["nx"] * case["ny"] * case["nz"], case["nx"] * case["ny"], case["h"], case["radius"]
    per_column = 0.0
    for k in range(case["nz"]):
        rho2 = r * r - ((k + 0.5) * h) ** 2
        per_column += max(0.0, math.pi * rho2 / (h * h)) if rho2 > 0 else 0.0
    return float(n), float(rays), rays * per_column


def work(case):
    """Bytes: the structure and the inputs once, the outputs once. Flops: five per entry
    (the residual's term) and one per neighbour in every proposal of an engine that sums a
    bit's terms anew; two per proposal (the move's energy from a carried field, and its
    test) in the engines that carry fields; two per entry of a sparse row."""
    kind = case["kind"]
    if kind in ("muon", "gravity", "muon_reference"):
        n, rays, nnz = gravity_work(case) if kind == "gravity" else muon_work(case)
        R = case["branches"]
        proposals = R * float(case["anneal"] + case["hold"])
        kept = R if kind == "gravity" or case.get("keep") else 0
        return {"bytes": 8 * nnz + 32 * n + 16 * rays + n * (9 + kept), "flops": proposals * (5 * nnz + 8 * n)}
    if kind == "energy":
        n, rays, nnz = muon_work(case)
        K = case["states"]
        return {"bytes": 8 * nnz + 32 * n + 16 * rays + K * n, "flops": K * (2 * nnz + 4 * rays + 8 * n)}
    if kind == "maxcut":
        n, m, R = case["n"], 0.5 * case["n"] * case["degree"], case["replicas"]
        return {"bytes": 16 * m + 8 * n + R * (n + 8.0), "flops": 2.0 * n * R * (case["anneal"] + case["hold"])}
    if kind == "qubo":
        degrees = [int(d) for d in case["degrees"].split(",")]
        lo, hi = case["n_lo"], case["n_hi"]
        n = (hi - lo) / math.log(hi / lo) if hi > lo else lo
        bits = case["instances"] * float(n)
        entries = bits * sum(degrees) / len(degrees)
        R = 0.5 * (case["r_lo"] + case["r_hi"])
        return {"bytes": 8 * entries + 8 * bits + R * bits, "flops": 2.0 * entries * R * case["sweeps"]}
    if kind == "dense":
        n, R = float(case["n"]), case["replicas"]
        full = case["sweeps"] // case["recompute"] if case["recompute"] else 0
        return {"bytes": 4 * n * n + 4 * n + R * (n + 8), "flops": R * (2.0 * n * case["sweeps"] + 2.0 * n * n * full)}
    # the energy and the weight of every state once
    return {"bytes": 8.0 * case["n"] * (case["n"] + 2), "flops": 4.0 * 2.0 ** case["n"]}


# ---- the outputs in 64 bits ----------------------------------------------------------------

def exact_energy(case, seed):
    P = muon_arrays(case, seed)
    X = branch_like_states(P, case["states"], seed)
    bit = np.repeat(np.arange(P.n_vars), np.diff(P.row_ptr))
    at = np.repeat(np.arange(P.n_vars), np.diff(P.nbr_ptr))
    a = P.a.astype(np.float64)
    data, prior = np.zeros(len(X)), np.zeros(len(X))
    for k, x in enumerate(X):
        r = np.bincount(P.ray, weights=a * x[bit], minlength=P.n_rays) - P.d
        data[k] = 0.5 * np.sum(P.w * r * r)
        # every pair stands in both bits' lists
        prior[k] = P.lam * 0.5 * np.count_nonzero(x[at] != x[P.nbr]) + P.kappa * np.count_nonzero(x)
    return dict(total=data + prior, data=data, prior=prior)


def exact_roi(case, seed):
    h, J = region(case, seed)
    n, beta = case["n"], case["beta"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    low = min(n, 22)

    def energies(field, bits):
        """E of every state of `bits` (bit i of the index = the i-th), fields `field`."""
        e = torch.zeros(1, dtype=torch.float64, device=dev)
        f = [torch.full((1,), float(v), dtype=torch.float64, device=dev) for v in field]
        for i, b in enumerate(bits):
            e = torch.cat([e, e + f[i]])
            f = [torch.cat([v, v + J[b, bits[j]]]) if j > i else v for j, v in enumerate(f)]
        return e

    lo, hi = list(range(low)), list(range(low, n))
    blocks = []
    for c in range(1 << len(hi)):
        on = [b for i, b in enumerate(hi) if (c >> i) & 1]
        base = sum(h[b] for b in on) + sum(J[a, b] for a in on for b in on if a < b)
        blocks.append((c, base, [h[b] + sum(J[b, q] for q in on) for b in lo]))
    e_min, s_min = math.inf, 0
    for c, base, field in blocks:
        e = energies(field, lo) + base
        i = int(torch.argmin(e))
        if float(e[i]) < e_min:
            e_min, s_min = float(e[i]), (c << low) | i
    z, marginal = 0.0, np.zeros(n)
    for c, base, field in blocks:
        w = torch.exp(-beta * (energies(field, lo) + (base - e_min)))
        s = float(w.sum())
        z += s
        for i in range(low):
            marginal[i] += float(w.view(-1, 2, 1 << i)[:, 1].sum())
        for i in range(len(hi)):
            if (c >> i) & 1:
                marginal[low + i] += s
    return dict(marginal=marginal / z, map_state=np.array([(s_min >> i) & 1 for i in range(n)], np.uint8),
                e_min=e_min, log_z=-beta * e_min + math.log(z), p_map=1.0 / z)


def exact(case, seed):
    if case["kind"] == "energy":
        return exact_energy(case, seed)
    if case["kind"] == "roi" and case["n"] <= 28:
        return exact_roi(case, seed)
    return None   # an anneal's outputs follow its random trajectory
