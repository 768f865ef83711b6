"""Performance cases of the recovery framework.

Each case is one call pattern of a user's program through the public entry
points: a problem given as host arrays (`cs`), a generated instance kept
resident (`Plan`), many independent instances in one launch (`Batch`), many
signals that share one matrix (`ManyRHS`) and the warm-start network (`MLP`).
A pass runs the call and returns what the caller is after: the recovered
vectors, the gradients or the scores, as host arrays.

Densities lie in the region where the algorithms recover the planted signal,
so the answer is well defined: the noise-free solution of every recovery is the
planted vector itself.
"""
import math

import numpy as np

import gaga_amd as ga

TOL = 1e-5
# Dense products with the matrix that a recovery at these densities needs at
# the least (its iterations, one gradient each).
PRODUCTS = 10

F, H = 8, 512  # the network: 8 features -> 512 -> 512 -> 1


def listed():
    return [
        # the smallest call: a given dense problem of 256 x 1024 (1 MB of host data), where
        # launches, allocations and barriers count
        {"name": "cs_gen_small", "kind": "cs", "alg": "NIHT", "ens": "gen", "m": 256, "n": 1024, "k": 20},
        # a given problem with sampled DCT rows (imaging-like), a ragged row count
        {"name": "cs_dct_medium", "kind": "cs", "alg": "CGIHT", "ens": "dct", "m": 5001, "n": 16384, "k": 300},
        # one dense instance at the size of the reference's single-problem workload
        {"name": "plan_gen_large", "kind": "plan", "alg": "CGIHT", "ens": "gen", "m": 2048, "n": 8192, "k": 205,
         "p": 0},
        # hard thresholding pursuit (a CG projection in every iteration) at odd sizes
        {"name": "plan_gen_htp_odd", "kind": "plan", "alg": "HTP", "ens": "gen", "m": 1001, "n": 5003, "k": 77,
         "p": 0},
        # the large sparse (expander-like) instance
        {"name": "plan_smv_large", "kind": "plan", "alg": "CGIHT", "ens": "smv", "m": 32768, "n": 262144,
         "k": 3277, "p": 7},
        # an ordinary sparse instance, odd sizes, the steepest-descent algorithm
        {"name": "plan_smv_odd", "kind": "plan", "alg": "NIHT", "ens": "smv", "m": 4999, "n": 20001, "k": 300,
         "p": 7},
        # the large DCT instance
        {"name": "plan_dct_large", "kind": "plan", "alg": "NIHT", "ens": "dct", "m": 131072, "n": 1048576,
         "k": 10000, "p": 0},
        # throughput: many equal dense instances in one launch with the tail schedule of the
        # benchmark, 34 GB of matrices
        {"name": "batch_gen_large", "kind": "batch", "alg": "CGIHT", "mix": "gen", "m": 2048, "n": 8192, "k": 205,
         "count": 512, "schedule": True},
        # an uneven batch: both ensembles and all sizes of the phase-transition sweep
        {"name": "batch_uneven", "kind": "batch", "alg": "CGIHT", "mix": "uneven", "m": 0, "n": 8192, "k": 0,
         "count": 256, "schedule": False},
        # many signals on one matrix, mixed precision, the benchmark's size
        {"name": "many_rhs_bf16", "kind": "mrhs", "precision": "bf16", "m": 4096, "n": 16384, "k": 400,
         "count": 512},
        # the FP8 form on a smaller matrix with a ragged number of signals
        {"name": "many_rhs_fp8_ragged", "kind": "mrhs", "precision": "fp8", "m": 1024, "n": 4096, "k": 60,
         "count": 200},
        # one training step's forward and backward of the network at its training batch
        {"name": "mlp_grad", "kind": "mlp", "batch": 8192, "train": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cs", "cs", "plan", "plan", "plan", "batch", "mrhs", "mlp"])
    rho = rng.uniform(0.02, 0.07)
    if kind in ("cs", "plan"):
        alg = rng.choice(["NIHT", "HTP", "CGIHT"])
        ens = rng.choice(["gen", "dct"] if kind == "cs" else ["gen", "smv", "dct"])
        delta = rng.uniform(0.2, 0.5)
        p = 0
        if ens == "gen":
            n = _log(rng, 700, 4096 if kind == "cs" else 9000)
            m = min(int(delta * n), 2500)
        elif ens == "smv":
            n, p = _log(rng, 4000, 262144), rng.choice([6, 7, 8, 9])
            m = int(min(delta, 0.25) * n)
        else:
            n = 2 ** rng.randint(11, 15 if kind == "cs" else 20)
            m = int(min(delta, 0.3) * n) | 1
        k = max(5, int(rho * m))
        c = {"kind": kind, "alg": alg, "ens": ens, "m": m, "n": n, "k": k}
        if kind == "plan":
            c["p"] = p
        return c
    if kind == "batch":
        if rng.random() < 0.5:
            return {"kind": "batch", "alg": rng.choice(["NIHT", "CGIHT"]), "mix": "uneven", "m": 0,
                    "n": rng.choice([4096, 8192]), "k": 0, "count": _log(rng, 16, 256), "schedule": False}
        n = _log(rng, 700, 8192)
        m = int(rng.uniform(0.25, 0.5) * n)
        count = max(4, min(_log(rng, 16, 512), int(2e9 / (m * n))))
        return {"kind": "batch", "alg": rng.choice(["NIHT", "CGIHT"]), "mix": "gen", "m": m, "n": n,
                "k": max(5, int(rho * m)), "count": count, "schedule": rng.random() < 0.5}
    if kind == "mrhs":
        m = 128 * _log(rng, 4, 32)
        n = max(1024, min(16384, m * rng.randint(2, 4) // 512 * 512))
        return {"kind": "mrhs", "precision": rng.choice(["bf16", "fp8"]), "m": m, "n": n,
                "k": max(10, int(rho * m)), "count": _log(rng, 16, 512)}
    return {"kind": "mlp", "batch": _log(rng, 100, 16384), "train": rng.random() < 0.6}


# ------------------------------------------------------------------ inputs --
def _sparse(rng, n, k):
    """A planted vector: k random signs on a random support."""
    x = np.zeros(n)
    x[rng.choice(n, k, replace=False)] = rng.choice([-1.0, 1.0], k)
    return x


def _dct2(x):
    """Orthonormal DCT-II in 64 bits by one FFT of the even-odd reordered input."""
    n = x.size
    v = np.concatenate([x[::2], x[1::2][::-1]])
    c = np.real(np.fft.fft(v) * np.exp(-0.5j * np.pi * np.arange(n) / n)) * math.sqrt(2.0 / n)
    c[0] *= math.sqrt(0.5)
    return c


def _given(case, seed):
    """(planted vector, y, matrix or sampled rows) of a given-problem call, host arrays."""
    rng = np.random.default_rng(seed)
    m, n, k = case["m"], case["n"], case["k"]
    x = _sparse(rng, n, k)
    if case["ens"] == "gen":
        A = (rng.standard_normal((n, m), dtype=np.float32) / np.float32(math.sqrt(m))).T  # column-major
        return x, (A.astype(np.float64) @ x).astype(np.float32), A
    rows = np.sort(rng.choice(n, m, replace=False))
    return x, _dct2(x)[rows].astype(np.float32), (rows + 1).astype(np.int32)


def _specs(case):
    """Instances of a batch: equal dense ones, or both ensembles over the sizes and
    undersampling rates of a phase-transition sweep."""
    if case["mix"] == "gen":
        return [dict(ens="gen", k=case["k"], m=case["m"], n=case["n"], instance=i) for i in range(case["count"])]
    out = []
    for i in range(case["count"]):
        n = case["n"] >> (i % 4)
        m = int(math.ceil((0.25 + 0.5 * ((i // 8) % 16) / 15) * n))
        k = max(4, int((0.03 + 0.05 * ((i // 128) % 4) / 3) * m))
        s = dict(ens="smv" if (i // 4) % 2 else "gen", n=n, m=m, k=k, instance=i)
        if s["ens"] == "smv":
            s["p"] = 7
        out.append(s)
    return out


def _net_inputs(case, seed):
    """Parameters of a network in training, features in their range, labels."""
    rng = np.random.default_rng(seed)
    par = np.zeros(F * H + H + H * H + H + H + 1, np.float32)
    o = 0
    for size, scale in ((F * H, math.sqrt(2 / F)), (H, 0.01), (H * H, math.sqrt(2 / H)), (H, 0.01),
                        (H, math.sqrt(1 / H)), (1, 0.01)):
        par[o:o + size] = rng.standard_normal(size) * scale
        o += size
    X = np.abs(rng.standard_normal((case["batch"], F))).astype(np.float32)
    X[:, 5], X[:, 6] = 0.25, 0.1
    X[:, 7] = np.minimum(np.log2(1 + X[:, 4]), 8) / 8
    return par, X, (rng.random(case["batch"]) < 0.3).astype(np.float32)


def _options(case, seed):
    o = {"tol": TOL, "seed": seed & 0x7FFFFFFF}
    if case["kind"] == "mrhs":
        o["vecDistribution"] = "gaussian"
    elif case.get("ens") == "smv":
        o["matrixEnsemble"] = "binary"
    return ga.options(**o)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "cs":
        _, y, M = _given(case, seed)
        return {"case": case, "y": y, "M": M, "opts": ga.options(tol=TOL)}
    if kind == "plan":
        return {"case": case, "h": ga.Plan(case["alg"], case["ens"], case["k"], case["m"], case["n"], case["p"],
                                           _options(case, seed))}
    if kind == "batch":
        o = {"tol": TOL, "seed": seed & 0x7FFFFFFF, "blockSize": 1024 if case["schedule"] else 512}
        B = ga.Batch(case["alg"], _specs(case), ga.options(**o))
        if case["schedule"]:
            B.schedule([1, 4, 8, 16, 32], [28, 8, 16, 32, 5000])
        elif case["mix"] == "uneven":
            B.configure(4, 512, max(1, case["count"] // 4))  # teams of 4 for the largest quarter
        return {"case": case, "h": B}
    if kind == "mrhs":
        return {"case": case, "h": ga.ManyRHS(case["m"], case["n"], case["k"], case["count"], case["precision"],
                                              _options(case, seed))}
    par, X, lab = _net_inputs(case, seed)
    net = ga.MLP(seed=1)
    net.set_params(par)
    return {"case": case, "h": net, "X": X, "lab": lab}


def run(state):
    case = state["case"]
    kind, h = case["kind"], state.get("h")
    if kind == "cs":
        if case["ens"] == "gen":
            return ga.cs(case["alg"], "gen", state["y"], state["M"], case["k"], state["opts"])[0]
        return ga.cs(case["alg"], "dct", state["y"], state["M"], case["k"], case["m"], case["n"],
                     state["opts"])[0]
    if kind == "plan":
        h.solve()
        return h.results()["x"]
    if kind == "batch":
        h.solve()
        return np.concatenate([h.x(i)[0] for i in range(h.count)])
    if kind == "mrhs":
        h.solve()
        return np.concatenate([h.x(s)[0] for s in range(h.count)])
    if case["train"]:
        return h.grad(state["X"], state["lab"], pos_w=2.0)[0]
    return h.scores(state["X"])


# ------------------------------------------------------------------- exact --
def _philox(i, stream, seed, inst):
    """Philox4x32-10 words 0 and 1 for counters (i, 0, stream, 0), key (seed, inst)."""
    M32 = np.uint64(0xFFFFFFFF)
    c = [i.astype(np.uint64), np.zeros(i.size, np.uint64), np.full(i.size, stream, np.uint64),
         np.zeros(i.size, np.uint64)]
    k0, k1 = seed & 0xFFFFFFFF, inst & 0xFFFFFFFF
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & M32, (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1),
             p0 & M32]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return c[0], c[1]


def _planted(n, k, seed, inst, gaussian=False):
    """The vector a generated instance plants: its support is the k indices with the
    smallest 64-bit keys of stream 1, its values come from stream 2."""
    a, b = _philox(np.arange(n), 1, seed, inst)
    s = np.argsort((a << np.uint64(32)) | b, kind="stable")[:k]
    a, b = _philox(s, 2, seed, inst)
    x = np.zeros(n)
    if gaussian:
        u, v = (a + 0.5) * 2.0 ** -32, (b + 0.5) * 2.0 ** -32
        x[s] = (np.sqrt(-2 * np.log(u)) * np.cos(2 * np.pi * v)).astype(np.float32)
    else:
        x[s] = np.where(a & np.uint64(1), 1.0, -1.0)
    return x


def _bf16(a):
    """The network's layer-2 operands are BF16 by design: round to nearest even."""
    u = np.asarray(a, np.float32).view(np.uint32).astype(np.uint64)
    u = (u + 0x7FFF + ((u >> np.uint64(16)) & np.uint64(1))) >> np.uint64(16)
    return (u.astype(np.uint32) << np.uint32(16)).view(np.float32).astype(np.float64)


def _network(case, seed):
    """Forward, and backward of the mean weighted cross-entropy, in 64 bits."""
    par, X, y = _net_inputs(case, seed)
    parts, o = [], 0
    for size in (F * H, H, H * H, H, H, 1):
        parts.append(par[o:o + size].astype(np.float64))
        o += size
    W1, b1, W2, b2, W3, b3 = parts
    W1, W2 = W1.reshape(H, F), _bf16(W2).reshape(H, H)
    X = X.astype(np.float64)
    h1 = _bf16(np.maximum(X @ W1.T + b1, 0))
    a2 = np.maximum(h1 @ W2.T + b2, 0)
    logit = a2 @ W3 + b3
    if not case["train"]:
        return logit
    dl = np.where(y > 0.5, 2.0, 1.0) * (1 / (1 + np.exp(-logit)) - y) / len(y)
    dz2 = np.where(a2 > 0, dl[:, None] * W3, 0)
    dz1 = np.where(h1 > 0, _bf16(dz2) @ W2, 0)
    return np.concatenate([(dz1.T @ X).ravel(), dz1.sum(0), (dz2.T @ h1).ravel(), dz2.sum(0), dl @ a2,
                           [dl.sum()]])


def exact(case, seed):
    kind = case["kind"]
    s = seed & 0x7FFFFFFF
    if kind == "cs":
        return _given(case, seed)[0]
    if kind == "plan":
        return _planted(case["n"], case["k"], s, 0)
    if kind == "batch":
        return np.concatenate([_planted(c["n"], c["k"], s, c["instance"]) for c in _specs(case)])
    if kind == "mrhs":
        return np.concatenate([_planted(case["n"], case["k"], s, 1 + q, True) for q in range(case["count"])])
    return _network(case, seed)


# -------------------------------------------------------------------- work --
def _matrix(ens, m, n, p):
    """(bytes, flops) of one product with the matrix: dense values, or sparse values and
    indices, or a transform."""
    if ens == "gen":
        return 4.0 * m * n, 2.0 * m * n
    if ens == "smv":
        return 8.0 * n * p + 4.0 * (m + n), 2.0 * n * p
    return 4.0 * n + 8.0 * m, 2.5 * n * math.log2(n)


def work(case):
    kind = case["kind"]
    if kind in ("cs", "plan"):
        b, f = _matrix(case["ens"], case["m"], case["n"], case.get("p", 0))
        return {"bytes": PRODUCTS * b, "flops": PRODUCTS * f}
    if kind == "batch":
        t = [_matrix(s["ens"], s["m"], s["n"], s.get("p", 0)) for s in _specs(case)]
        return {"bytes": PRODUCTS * sum(b for b, _ in t), "flops": PRODUCTS * sum(f for _, f in t)}
    if kind == "mrhs":
        m, n, c = case["m"], case["n"], case["count"]
        e = 2.0 if case["precision"] == "bf16" else 1.0
        return {"bytes": 3 * PRODUCTS * e * (m * n + c * (m + n)), "flops": 3 * PRODUCTS * 2.0 * m * n * c}
    B = case["batch"]
    return {"bytes": 4.0 * (B * (F + 1) + 2 * H * H), "flops": (6.0 if case["train"] else 2.0) * B * H * H}
