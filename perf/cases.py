"""The work a user of this library has it do, as measurable cases.

Every case goes through the package's public entry points: factorizations of a resident matrix
(Job.run), the two half-steps a driver calls by itself (Job.update_H / Job.update_W), the rank
sweep, the serving loop, the out-of-core job and the quality figures of a finished
factorization.  Sizes are those of the benchmark, the tests and the request stream; listed()
says for each case what it stands for, draw() gives more of the same ranges.

A pass starts every factorization from its seed's random factors, as a program that tries
several starts does, runs a fixed number of iterations (the stop rule is out of reach, so that
the work does not depend on rounding) and fetches the factors.  exact() repeats the updates in
64 bits with plain torch.
"""
import importlib.util
import math
import pathlib
import random
import sys

import numpy as np
import torch

ROOT = pathlib.Path(__file__).resolve().parent.parent
NEVER = 1_000_000_000     # unchanged tests needed to stop: more than any run performs
T = 10                    # iterations between convergence tests (the default)
FLT_MIN = 1.17549435e-38  # lower clamp of the factors at every test


def _package():
    name = "bionmf_gpu_amd"
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(name, ROOT / "bionmf-gpu_amd" / "__init__.py")
        sys.modules[name] = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(sys.modules[name])
    return sys.modules[name]


# ------------------------------------------------------------------------------ the cases

def listed():
    return [
        # the half-steps called one by one, as a driver of the reference's style does, on the
        # smallest matrix of the smoke test: nothing but launches and latency
        {"name": "half_steps_tiny", "op": "half", "n": 600, "m": 40, "k": 3, "data": "lognormal", "iters": 20},
        # gene expression of a few samples: the benchmark's small job
        {"name": "small_job", "op": "run", "n": 5000, "m": 38, "k": 3, "data": "lognormal", "iters": 200, "path": 0},
        # many rows of very few columns (the vector-ALU kernels)
        {"name": "narrow", "op": "run", "n": 60000, "m": 20, "k": 4, "data": "lognormal", "iters": 100, "path": 0},
        # an ordinary matrix with no even size in it
        {"name": "ragged_mid", "op": "run", "n": 7013, "m": 333, "k": 7, "data": "planted", "iters": 100, "path": 0},
        # the benchmark's headline job, shortened
        {"name": "headline", "op": "run", "n": 20000, "m": 1000, "k": 16, "data": "planted", "iters": 100, "path": 0},
        # the same matrix at the largest rank that runs in FP32 by itself
        {"name": "rank32", "op": "run", "n": 20000, "m": 1000, "k": 32, "data": "planted", "iters": 60, "path": 0},
        # the benchmark's dense rank, with the default BF16 contractions ...
        {"name": "dense_bf16", "op": "run", "n": 50000, "m": 2000, "k": 64, "data": "planted", "iters": 20, "path": 0},
        # ... and in FP32 as the drop-in layer runs every rank
        {"name": "dense_fp32", "op": "run", "n": 50000, "m": 2000, "k": 64, "data": "planted", "iters": 10, "path": 2},
        # the benchmark's rank sweep with fewer restarts, all jobs batched
        {"name": "sweep", "op": "sweep", "n": 5000, "m": 200, "k_lo": 2, "k_hi": 10, "restarts": 6, "iters": 200},
        # a burst of uneven requests to the serving loop
        {"name": "serve", "op": "serve", "mix": 11, "count": 8, "n_hi": 20000, "m_hi": 1500, "restarts": 5, "iters": 100},
        # the quality figures (Frobenius, KL) of a finished factorization
        {"name": "quality", "op": "quality", "n": 20000, "m": 1000, "k": 16, "data": "planted"},
        # V kept in (pinned) host memory and streamed once per iteration
        {"name": "streamed", "op": "streamed", "n": 20000, "m": 1000, "k": 16, "data": "planted", "iters": 4,
         "block_rows": 4096},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["run", "run", "run", "run", "run", "run", "half", "quality", "sweep", "serve", "streamed"])
    data = rng.choice(["planted", "lognormal"])
    if op == "serve":
        return {"op": op, "mix": rng.randrange(1 << 20), "count": rng.randint(4, 8),
                "n_hi": _log_uniform(rng, 4000, 20000), "m_hi": _log_uniform(rng, 200, 1500),
                "restarts": rng.randint(2, 4), "iters": 10 * rng.randint(4, 8)}
    if op == "sweep":
        lo = rng.randint(2, 8)
        return {"op": op, "n": _log_uniform(rng, 1000, 5000), "m": _log_uniform(rng, 40, 200), "k_lo": lo,
                "k_hi": lo + rng.randint(1, 4), "restarts": rng.randint(2, 6), "iters": 10 * rng.randint(5, 15)}
    while True:
        n, m = _log_uniform(rng, 500, 60000), _log_uniform(rng, 20, 3000)
        if n * m <= 60_000_000:
            break
    k = rng.randint(2, min(64 if rng.random() < 0.25 else 32, m))
    if op == "quality":
        return {"op": op, "n": n, "m": m, "k": k, "data": data}
    if op == "streamed":
        return {"op": op, "n": n, "m": m, "k": k, "data": data, "iters": rng.randint(2, 4),
                "block_rows": 64 * rng.randint(16, 64)}
    if op == "half":
        n, m = min(n, 5000), min(m, 1000)
        return {"op": op, "n": n, "m": m, "k": k, "data": data, "iters": rng.randint(10, 30)}
    iters = 10 * max(1, min(10, int(1.5e10 / (10.0 * n * m * max(k, 16)))))
    return {"op": op, "n": n, "m": m, "k": k, "data": data, "iters": iters,
            "path": 2 if k > 32 and rng.random() < 0.5 else 0}


def _requests(case, seed):
    """The serving burst: the sizes follow from the case, the matrices' seeds from <seed>."""
    rng = random.Random(case["mix"])
    out = []
    for i in range(case["count"]):
        n, m = _log_uniform(rng, 1000, case["n_hi"]), _log_uniform(rng, 20, case["m_hi"])
        k = rng.randint(2, min(32, m))
        out.append((n, m, k, rng.randint(1, case["restarts"]), seed * 1000 + i, 0.0))
    return out


def work(case):
    """V once per iteration (once for the quality figures), both factors in and out, and the
    four contractions of an iteration."""
    def one(n, m, k, iters):
        return {"bytes": 4.0 * iters * (n * m + 2 * n * k + 2 * m * k), "flops": 8.0 * iters * n * m * k}
    if case["op"] == "sweep":
        parts = [one(case["n"], case["m"], k, case["iters"]) for k in range(case["k_lo"], case["k_hi"] + 1)
                 for _ in range(case["restarts"])]
    elif case["op"] == "serve":
        parts = [one(n, m, k, case["iters"]) for n, m, k, r, _, _ in _requests(case, 0) for _ in range(r)]
    elif case["op"] == "quality":
        n, m, k = case["n"], case["m"], case["k"]
        parts = [{"bytes": 4.0 * (n * m + n * k + m * k), "flops": 2.0 * n * m * k}]
    else:
        parts = [one(case["n"], case["m"], case["k"], case["iters"])]
    return {"bytes": sum(p["bytes"] for p in parts), "flops": sum(p["flops"] for p in parts)}


# ------------------------------------------------------------------------------ inputs

def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _matrix(case, seed):
    """V (n x m float32, on _device()): a planted rank-limited matrix under lognormal noise, or
    lognormal expression values."""
    dev = _device()
    gen = torch.Generator(device=dev).manual_seed(seed)
    n, m = case["n"], case["m"]
    if case["data"] == "lognormal":
        return torch.exp(5.0 + 1.5 * torch.randn(n, m, device=dev, generator=gen))
    rank = max(2, min(48, n, m, case.get("k", 6) * 3 // 4 if case.get("k", 6) > 32 else case.get("k", 6)))
    W = torch.empty(n, rank, device=dev).exponential_(1.0, generator=gen)
    H = torch.empty(m, rank, device=dev).exponential_(1.0, generator=gen)
    return (W @ H.T) * torch.exp(0.3 * torch.randn(n, m, device=dev, generator=gen))


def _finished_factors(case, seed):
    """Factors as a finished factorization leaves them: of V's scale, some entries near zero."""
    dev = _device()
    gen = torch.Generator(device=dev).manual_seed(seed + 77)
    W = torch.empty(case["n"], case["k"], device=dev).exponential_(1.0, generator=gen) + 1e-6
    H = torch.empty(case["m"], case["k"], device=dev).exponential_(1.0, generator=gen) + 1e-6
    scale = 457.0 / case["k"] if case["data"] == "lognormal" else 1.0
    return W * scale, H


def prepare(case, seed):
    nmfk = _package()
    state = {"case": case, "seed": seed, "nmfk": nmfk}
    if case["op"] == "serve":
        state["requests"] = _requests(case, seed)
        return state
    n, m = case["n"], case["m"]
    V = _matrix(dict(case, data="planted", k=6) if case["op"] == "sweep" else case, seed).cpu().numpy()
    if case["op"] == "streamed":
        state["job"] = nmfk.Job.streamed(V, case["k"], case["block_rows"], pinned=True)
        return state
    job = state["job"] = nmfk.Job(n, m, case.get("k", 1))
    job.set_V(V)
    if case.get("path"):
        job.set_kernel_path(case["path"])
    if case["op"] == "quality":
        W, H = _finished_factors(case, seed)
        job.set_WH(W.cpu().numpy(), H.cpu().numpy())
    return state


# ------------------------------------------------------------------------------ one pass

def run(state):
    case, seed, nmfk = state["case"], state["seed"], state["nmfk"]
    if case["op"] == "serve":
        requests = state["requests"]
        res, _ = nmfk.serve(requests, nIters=case["iters"], niter_test_conv=T, stop_threshold=NEVER, detail=True,
                            factors_of=range(len(requests)))
        runs = [r for q in res for r in q["restarts"]]
        return {"W": np.concatenate([r["W"].ravel() for r in runs]),
                "H": np.concatenate([r["H"].ravel() for r in runs]),
                "kl": np.array([r["kl"] for r in runs], np.float32)}
    job = state["job"]
    if case["op"] == "sweep":
        r = nmfk.sweep(job, range(case["k_lo"], case["k_hi"] + 1), case["restarts"], seed, nIters=case["iters"],
                       niter_test_conv=T, stop_threshold=NEVER, plan_target=16, want_factors=True)
        return {"W": np.concatenate([W.ravel() for W, _ in r["factors"]]),
                "H": np.concatenate([H.ravel() for _, H in r["factors"]])}
    if case["op"] == "quality":
        return np.array(job.dot_kl())
    job.init_random(seed)
    if case["op"] == "half":
        for i in range(case["iters"]):
            job.update_H()
            job.update_W()
            if (i + 1) % T == 0:
                job.adjust()
    else:
        job.run(case["iters"], T, NEVER)
    return {"W": job.get_W(), "H": job.get_H()}


# ------------------------------------------------------------------------------ in 64 bits

def _philox(seed, tag, block, dev):
    """Philox4x32-10 (Salmon et al., SC'11) of the counters (block, tag, domain): four int64
    tensors holding 32-bit words."""
    low = 0xFFFFFFFF
    block = block.to(dev)
    c = [block & low, (block >> 32) & low, torch.full_like(block, tag), torch.full_like(block, 0x4E4D4621)]
    k0, k1 = seed & low, (seed >> 32) & low
    for _ in range(10):
        p0, p1 = 0xD2511F53 * c[0], 0xCD9E8D57 * c[2]
        c = [((p1 >> 32) & low) ^ c[1] ^ k0, p1 & low, ((p0 >> 32) & low) ^ c[3] ^ k1, p0 & low]
        k0, k1 = (k0 + 0x9E3779B9) & low, (k1 + 0xBB67AE85) & low
    return c


def _start(rows, k, seed, tag, dev):
    """The random factor of a seed: uniform (0, 1] in 24 bits."""
    count = rows * k
    words = torch.stack(_philox(seed, tag, torch.arange((count + 3) // 4), dev), 1).reshape(-1)[:count]
    return (((words >> 8) + 1).double() / 16777216.0).reshape(rows, k)


def _lognormal(n, m, seed, dev):
    """The serving loop's input matrix of a seed: exp(N(5, 1.5^2)), Box-Muller on 53-bit uniforms."""
    w = _philox(seed, 0x100, torch.arange(n * m), dev)
    u1, u2 = (((((a >> 5) << 26) | (b >> 6)).double() + 1.0) / 9007199254740992.0 for a, b in ((w[0], w[1]), (w[2], w[3])))
    z = torch.sqrt(-2.0 * torch.log(u1)) * torch.cos(2.0 * math.pi * u2)
    return torch.exp(5.0 + 1.5 * z).float().double().reshape(n, m)


def _seed_of(base, k, restart):
    """splitmix64's finaliser of base ^ (k << 32 | restart)."""
    x = (base ^ ((k << 32) | restart)) & (2 ** 64 - 1)
    x = (x + 0x9E3779B97F4A7C15) & (2 ** 64 - 1)
    x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & (2 ** 64 - 1)
    x = ((x ^ (x >> 27)) * 0x94D049BB133111EB) & (2 ** 64 - 1)
    return x ^ (x >> 31)


def _factorize(V, k, seed, iters):
    W, H = _start(V.shape[0], k, seed, 0, V.device), _start(V.shape[1], k, seed, 1, V.device)
    for i in range(iters):
        H = H * ((V / (W @ H.T)).T @ W) / W.sum(0)
        W = W * ((V / (W @ H.T)) @ H) / H.sum(0)
        if (i + 1) % T == 0:
            W, H = W.clamp_min(FLT_MIN), H.clamp_min(FLT_MIN)
    return W, H


def _quality(V, W, H):
    WH = W @ H.T
    kl = torch.where(V > 0, V * torch.log(V / WH), torch.zeros_like(V)) - V + WH
    return [float((V * V).sum()), float(((V - WH) ** 2).sum()), float(kl.sum())]


def exact(case, seed):
    dev = _device()
    if dev == "cpu" and work(case)["flops"] > 2e10:
        return None
    if case["op"] == "serve":
        done, kl = [], []
        for n, m, k, restarts, s, _ in _requests(case, seed):
            V = _lognormal(n, m, s, dev)
            for r in range(restarts):
                done.append(_factorize(V, k, _seed_of(s, k, r), case["iters"]))
                kl.append(_quality(V, *done[-1])[2])
        return {"W": torch.cat([W.reshape(-1) for W, _ in done]), "H": torch.cat([H.reshape(-1) for _, H in done]),
                "kl": torch.tensor(kl, dtype=torch.float64)}
    V = _matrix(dict(case, data="planted", k=6) if case["op"] == "sweep" else case, seed).double()
    if case["op"] == "sweep":
        done = [_factorize(V, k, _seed_of(seed, k, r), case["iters"])
                for k in range(case["k_lo"], case["k_hi"] + 1) for r in range(case["restarts"])]
        return {"W": torch.cat([W.reshape(-1) for W, _ in done]), "H": torch.cat([H.reshape(-1) for _, H in done])}
    if case["op"] == "quality":
        W, H = _finished_factors(case, seed)
        return torch.tensor(_quality(V, W.double(), H.double()), dtype=torch.float64)
    W, H = _factorize(V, case["k"], seed, case["iters"])
    return {"W": W, "H": H}
