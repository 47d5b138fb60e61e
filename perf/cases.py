"""The calls that programs using culip_amd spend their time in, as cases to time.

A case is a dict of plain values; `prepare` makes what the program holds
before the call, `run` is one pass through the public entry points. The
systems are the KKT generator's (H with `o` off-diagonals per row, A with `c`
entries per column, m dual rows), ordered by block colouring with blocks of at
most `B` rows, the sizes those of the benchmark and the tests.

Operations (`op`):
  spmv      y = K x with the assembled matrix
  operator  y = K x without assembling K (H and A as CSR)
  apply     the preconditioner on a vector: U' solve, D solve, U solve
  refactor  new values of a resident pattern into the factor, then one
            application of it
  solve     refactor and SQMR to a true relative residual of 1e-8
  batch     many systems refactored and solved together
  serve     host requests over resident patterns through the request loop
"""
import concurrent.futures
import functools
import math

import numpy as np
import torch

import culip_amd as ca

TOL = 1e-8


def listed():
    return [
        # one operator product at the size of the large benchmark system: the
        # inner step of any Krylov method over an assembled KKT matrix
        dict(name="spmv-400k", op="spmv", n=400000, m=150000, o=6, c=4),
        # the same without assembling K, as an interior-point code that keeps
        # H and A apart does; sizes no multiple of a tile
        dict(name="operator-77k", op="operator", n=77777, m=31111, o=4, c=3),
        # the smallest call: one preconditioner application on a system of a
        # few thousand rows, all latency
        dict(name="apply-2k", op="apply", n=2000, m=800, o=4, c=3, B=32, prec="f64",
             algo="single", sweeps=0),
        # exact triangular solves at the large size
        dict(name="apply-400k", op="apply", n=400000, m=150000, o=6, c=4, B=32, prec="f64",
             algo="single", sweeps=0),
        # block-Jacobi solves with an FP32 factor, the serving preconditioner
        dict(name="apply-50k-jacobi-f32", op="apply", n=50001, m=20003, o=4, c=3, B=32,
             prec="f32", algo="jacobi", sweeps=2),
        # new values of a small pattern (the step of a small interior-point
        # solve): many launches over little work
        dict(name="refactor-2k", op="refactor", n=2000, m=800, o=4, c=3, B=32, prec="f64",
             pivoting="static"),
        # numeric Bunch-Kaufman pivots, for matrices without static ones
        dict(name="refactor-33k-bk", op="refactor", n=33333, m=12345, o=4, c=3, B=32,
             prec="f64", pivoting="bk"),
        # the large pattern's refactor
        dict(name="refactor-400k", op="refactor", n=400000, m=150000, o=6, c=4, B=32,
             prec="f64", pivoting="static"),
        # a whole interior-point step at the reference driver's small size
        dict(name="solve-2k", op="solve", n=2000, m=800, o=4, c=3, B=32, prec="f64",
             algo="single", sweeps=0),
        # and at the large one, the benchmark's step
        dict(name="solve-400k", op="solve", n=400000, m=150000, o=6, c=4, B=32, prec="f64",
             algo="single", sweeps=0),
        # independent systems of 1,000 to 40,000 primal rows solved together
        # (FP32 factors, two block-Jacobi sweeps)
        dict(name="batch-256", op="batch", count=256, lo=1000, hi=40000, B=8, prec="f32",
             sweeps=2, first=0),
        # a burst of requests with fresh barrier weights over four patterns
        dict(name="serve-24", op="serve", patterns=4, requests=24, lo=5000, hi=60000, B=32,
             prec="f32", sweeps=2, slots=4, first=500),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["spmv", "operator", "apply", "refactor", "solve", "apply", "refactor",
                     "solve", "batch", "serve"])
    if op == "batch":
        return dict(op=op, count=rng.randint(4, 96), lo=1000, hi=_log(rng, 4000, 40000),
                    B=rng.choice([8, 16, 32]), prec=rng.choice(["f32", "f64"]),
                    sweeps=rng.choice([2, 3]), first=rng.randint(0, 400))
    if op == "serve":
        return dict(op=op, patterns=rng.randint(1, 4), requests=rng.randint(2, 20), lo=2000,
                    hi=_log(rng, 5000, 50000), B=rng.choice([16, 32]),
                    prec=rng.choice(["f32", "f64"]), sweeps=rng.choice([2, 3]), slots=4,
                    first=rng.randint(0, 900))
    n = _log(rng, 1500, 300000)
    case = dict(op=op, n=n, m=int(n * rng.uniform(0.3, 0.45)), o=rng.choice([4, 6]),
                c=rng.choice([3, 4]))
    if op in ("spmv", "operator"):
        return case
    case.update(B=rng.choice([8, 16, 32]), prec=rng.choice(["f64", "f64", "f32"]))
    if op == "refactor":
        case["pivoting"] = rng.choice(["static", "static", "static", "bk", "rook"])
    else:
        case["algo"] = rng.choice(["single", "single", "levels", "jacobi"])
        case["sweeps"] = rng.choice([2, 3]) if case["algo"] == "jacobi" else 0
    return case


# --------------------------------------------------------------------------
# inputs

@functools.lru_cache(maxsize=400)
def _system(n, m, o, c, pattern, B):
    """(KKT, Prep or None) of a pattern; values follow from the seed later."""
    k = ca.KKT(n, m, o, c, seed=pattern)
    p = ca.Prep(k.row_ptr, k.col, k.val, n, B, ca.ORDER_BLOCK_COLOR) if B else None
    return k, p


def _product(row_ptr, col, val, x, dtype=np.float64):
    """K x on the host (every row of K has an entry)."""
    return np.add.reduceat(val.astype(dtype) * x.astype(dtype)[col], row_ptr[:-1])


def _values(k, p, seed, weights):
    """K's values with barrier weights drawn from the seed, in the order of p."""
    v = k.barrier_values(weights[0], weights[1], seed=seed)
    return v if p is None else p.permute_values(v)


MILD = (1e-2, 1.0)        # a step of a well-centred interior-point iteration
BARRIER = (1e-4, 1e4)     # fresh weights of unrelated requests


def _truth(n, seed):
    """The solution a linear system of n rows is set up to have."""
    return np.random.default_rng(seed).standard_normal(n)


def _many(case):
    """(pattern seed, n) of a batch's or a server's systems, spread over the
    logarithm of their range."""
    cnt = case["count"] if case["op"] == "batch" else case["patterns"]
    lo, hi = math.log(case["lo"]), math.log(case["hi"])
    return [(case["first"] + i,
             int(round(math.exp(lo + (hi - lo) * ((i * 0.6180339887498949) % 1.0)))))
            for i in range(cnt)]


def _many_systems(case):
    sizes = _many(case)
    with concurrent.futures.ThreadPoolExecutor(8) as ex:
        return list(ex.map(lambda s: _system(s[1], int(0.4 * s[1]), 4, 3, s[0], case["B"]),
                           sizes))


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _split(k):
    """H and A of the generator's K = [[H, A'], [A, -delta I]], as CSR."""
    n, N = k.n, k.N
    rows = np.repeat(np.arange(N), np.diff(k.row_ptr))
    h = (rows < n) & (k.col < n)
    a = (rows >= n) & (k.col < n)
    d = (rows >= n) & (k.col >= n)

    def csr(mask, first, count):
        rp = np.zeros(count + 1, np.int64)
        np.cumsum(np.bincount(rows[mask] - first, minlength=count), out=rp[1:])
        return rp.astype(np.int32), k.col[mask], np.flatnonzero(mask)
    return csr(h, 0, n), csr(a, n, N - n), float(k.val[d][0]) if d.any() else 0.0


def prepare(case, seed):
    op = case["op"]
    if op == "batch":
        systems = _many_systems(case)
        bt = ca.Batch(prec=case["prec"], jacobi_sweeps=case["sweeps"], tol=TOL)
        # systems are numbered in the order they are added
        for _, p in systems:
            bt.add(p.row_ptr, p.col, p.val, p.piv_starts, p.block_starts)
        vals = [_values(k, p, seed + i, MILD) for i, (k, p) in enumerate(systems)]
        rhs = [_product(p.row_ptr, p.col, v, _truth(k.N, seed + i))
               for i, ((k, p), v) in enumerate(zip(systems, vals))]
        return dict(op=op, batch=bt, vals=[_dev(v) for v in vals], rhs=[_dev(b) for b in rhs])
    if op == "serve":
        systems = _many_systems(case)
        sv = ca.Server(slots=case["slots"], prec=case["prec"], tol=TOL, max_it=3000,
                       true_residual_period=20, max_restarts=10, solve_algorithm="jacobi",
                       jacobi_sweeps=case["sweeps"], equilibrate_sweeps=8, graphs=True)
        ids = [sv.add_pattern(p.row_ptr, p.col, p.val, p.piv_starts, p.block_starts)
               for _, p in systems]
        reqs = []
        for r in range(case["requests"]):
            k, p = systems[r % len(systems)]
            v = _values(k, p, seed + r, BARRIER)
            reqs.append((ids[r % len(ids)], v, _product(p.row_ptr, p.col, v,
                                                        _truth(k.N, seed + r))))
        return dict(op=op, server=sv, requests=reqs)

    n, m, o, c = case["n"], case["m"], case["o"], case["c"]
    if op in ("spmv", "operator"):
        k, _ = _system(n, m, o, c, 0, 0)
        val = _values(k, None, seed, BARRIER)
        if op == "spmv":
            A = ca.CSRMatrixSPMV(k.row_ptr, k.col, val)
        else:
            (hp, hc, hi), (ap, ac, ai), delta = _split(k)
            A = ca.AugmentedMatrixSPMV(ap, ac, val[ai], n, delta=delta,
                                       ix=np.arange(m, dtype=np.int32), H=(hp, hc, val[hi]))
        x = _dev(_truth(k.N, seed))
        return dict(op=op, A=A, x=x, y=torch.zeros_like(x))

    k, p = _system(n, m, o, c, 0, case["B"])
    val = _values(k, p, seed, BARRIER if op == "refactor" else MILD)
    g = ca.BlockiLDLt(p.row_ptr, p.col, val, p.piv_starts, p.block_starts, case["prec"])
    if op == "refactor":
        g.set_pivoting(case["pivoting"])
    else:
        g.set_solve_algorithm(case["algo"], case["sweeps"])
    g.compute(0, 1.0, 1e-4)
    st = dict(op=op, g=g)
    truth = _truth(k.N, seed)
    if op == "solve":
        st["A"] = ca.CSRMatrixSPMV(p.row_ptr, p.col, val)
        st["sqmr"] = ca.SQMR(st["A"], TOL, 1000, g, true_residual_period=20, max_restarts=10)
        st["vals"] = _dev(val)
        st["b"] = _dev(_product(p.row_ptr, p.col, val, truth))
        st["x"] = torch.zeros_like(st["b"])
        return st
    if op == "refactor":
        st["vals"] = _dev(val)
    st["b"] = _dev(truth)
    st["x"] = [torch.zeros_like(st["b"]) for _ in range(3)]
    return st


def _apply(g, b, x):
    """x = (U' \\ b, D \\ that, U \\ that): M \\ b with its two half steps."""
    g.solve_left(b, x[0])
    g.solve_middle(x[0], x[1])
    g.solve_right(x[1], x[2])
    return x


def run(state):
    op = state["op"]
    if op in ("spmv", "operator"):
        state["A"].multiply(state["x"], state["y"])
        return state["y"]
    if op == "apply":
        return _apply(state["g"], state["b"], state["x"])
    if op == "refactor":
        state["g"].refactor(state["vals"], 1e-4)
        return _apply(state["g"], state["b"], state["x"])
    if op == "solve":
        state["g"].refactor(state["vals"], 1e-4)
        state["sqmr"].solve(state["b"], state["x"])
        return state["x"]
    if op == "batch":
        xs, _ = state["batch"].solve(state["vals"], state["rhs"])
        return torch.cat(xs)
    sv = state["server"]
    ids = [sv.submit(*r) for r in state["requests"]]
    return [sv.wait(i)[0] for i in ids]


# --------------------------------------------------------------------------
# what a pass cannot do without

ITERATIONS = 60   # SQMR iterations such systems take (40 to 100)


def _counts(n, m, o, c):
    """rows and entries of K"""
    return n + m, n * (1 + o) + 2 * c * n + m


def _factor_bytes(N, nnz, prec):
    """one pass over U (upper entries and their columns) and D"""
    return (nnz + N) // 2 * (4 + (4 if prec == "f32" else 8)) + 8 * N


def _refactor_bytes(N, nnz, prec):
    """K's values and columns in, U and D out"""
    return 12 * nnz + 4 * N + _factor_bytes(N, nnz, prec)


def _spmv_bytes(N, nnz):
    return 12 * nnz + 4 * (N + 1) + 16 * N


def _solve_work(N, nnz, prec):
    it = _spmv_bytes(N, nnz) + 2 * _factor_bytes(N, nnz, prec) + 8 * 12 * N
    return {"bytes": _refactor_bytes(N, nnz, prec) + ITERATIONS * it,
            "flops": 4 * nnz + ITERATIONS * (4 * nnz + 20 * N)}


def work(case):
    op = case["op"]
    if op in ("batch", "serve"):
        sizes = [n for _, n in _many(case)]
        if op == "serve":
            sizes = [sizes[r % len(sizes)] for r in range(case["requests"])]
        each = [_solve_work(*_counts(n, int(0.4 * n), 4, 3), case["prec"]) for n in sizes]
        return {key: sum(e[key] for e in each) for key in ("bytes", "flops")}
    N, nnz = _counts(case["n"], case["m"], case["o"], case["c"])
    if op == "spmv":
        return {"bytes": _spmv_bytes(N, nnz), "flops": 2 * nnz}
    if op == "operator":
        # A once for each of its two products, H once
        return {"bytes": _spmv_bytes(N, nnz), "flops": 2 * nnz}
    apply_bytes = 2 * _factor_bytes(N, nnz, case["prec"]) + 8 * 6 * N
    if op == "apply":
        return {"bytes": apply_bytes, "flops": 2 * nnz + 8 * N}
    if op == "refactor":
        return {"bytes": _refactor_bytes(N, nnz, case["prec"]) + apply_bytes,
                "flops": 6 * nnz + 8 * N}
    return _solve_work(N, nnz, case["prec"])


# --------------------------------------------------------------------------
# reference values

def exact(case, seed):
    op = case["op"]
    if op in ("apply", "refactor"):
        # an incomplete factor is defined by the library's own dropping
        # rules: nothing outside it says what its application gives
        return None
    if op == "batch":
        return np.concatenate([_truth(n + int(0.4 * n), seed + i)
                               for i, (_, n) in enumerate(_many(case))])
    if op == "serve":
        sizes = [n for _, n in _many(case)]
        return [_truth(sizes[r % len(sizes)] + int(0.4 * sizes[r % len(sizes)]), seed + r)
                for r in range(case["requests"])]
    n, m = case["n"], case["m"]
    if op == "solve":
        return _truth(n + m, seed)   # the right-hand side is K times it
    k, _ = _system(n, m, case["o"], case["c"], 0, 0)
    val = _values(k, None, seed, BARRIER)
    return _product(k.row_ptr, k.col, val, _truth(k.N, seed), np.longdouble).astype(np.float64)
