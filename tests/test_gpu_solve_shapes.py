"""The solve kernels at the sizes where their forms end. Batched Jacobi sweeps
(two block rows per pass up to 64 entries, 32 in the inverse, else one) against
the same systems alone; single-launch against per-level solves; SQMR runs of
every length against each other, whatever the check period. Equal bits
throughout: every form keeps the order of operations."""
import numpy as np
import pytest

import culip_amd as ca
import oracle_lib as ol
from conftest import sym_problem

pytestmark = pytest.mark.gpu


def _kkt(n, m, o, c, B, seed=5):
    k = ca.KKT(n, m, o, c, seed=seed)
    p = ca.Prep(k.row_ptr, k.col, k.val, n, B, ca.ORDER_BLOCK_COLOR)
    return (p.row_ptr, p.col, p.val), p.piv_starts, p.block_starts


def _problem(kind):
    """kind: (n, m, overlap, coupling, block height) of a KKT system,
    (blocks, largest height, density) of a random one with 2x2 pivots, or the
    number of rows of a diagonal matrix."""
    if isinstance(kind, int):
        i = np.arange(kind, dtype=np.int32)
        bs = np.arange(0, kind, 8, dtype=np.int32)
        return (np.arange(kind + 1, dtype=np.int32), i, 1.0 + i.astype(float)), i, bs
    if len(kind) == 3:
        csr, piv, bs, _ = sym_problem(n_blocks=kind[0], bmax=kind[1], density=kind[2],
                                      seed=kind[0])
        return csr, piv, bs
    return _kkt(*kind)


SHAPES = [
    (900, 361, 4, 3, 1), (900, 361, 4, 3, 8), (1203, 480, 6, 4, 16), (2000, 801, 4, 3, 32),
    (41, 4, 0.06), (41, 4, 0.12), (43, 4, 0.25), (23, 12, 0.08), (15, 32, 0.1), (1, 32, 0.3),
    1, 65,
]


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_batched_sweeps_equal_alone(hip_device, prec):
    import torch
    systems = [_problem(s) for s in SHAPES]
    rng = np.random.default_rng(3)
    rhs = [rng.normal(size=s[0][0].size - 1) for s in systems]
    bt = ca.Batch(prec=prec, tol=1e-14, max_it=7, true_residual_period=3, max_restarts=0,
                  jacobi_sweeps=3)
    for csr, piv, bs in systems:
        bt.add(*csr, piv, bs)
    xs, res = bt.solve([csr[2] for csr, _, _ in systems], rhs)
    bt.close()
    for i, ((csr, piv, bs), b) in enumerate(zip(systems, rhs)):
        g = ca.BlockiLDLt(*csr, piv, bs, prec)
        g.compute(0, 1.0, 1e-4)
        g.set_solve_algorithm("jacobi", 3)
        q = ca.SQMR(ca.CSRMatrixSPMV(*csr), 1e-14, 7, g, true_residual_period=3, max_restarts=0)
        x = torch.zeros(b.size, dtype=torch.float64, device=hip_device)
        q.solve(torch.tensor(b, device=hip_device), x)
        assert np.array_equal(x.cpu().numpy(), xs[i], equal_nan=True), SHAPES[i]
        assert q.result["iterations"] == res[i]["iterations"], SHAPES[i]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("shape", SHAPES)
def test_single_launch_equals_levels(hip_device, shape, prec):
    import torch
    csr, piv, bs = _problem(shape)
    g = ca.BlockiLDLt(*csr, piv, bs, prec)
    g.compute(0, 1.0, 1e-4)
    o = ol.OracleBildlt(*csr, piv, bs, "f" if prec == "f32" else "d")
    o.set_pivot_precision("f64")
    o.symbolic(0, 1.0)
    o.factor(1e-4)
    b = np.random.default_rng(9).normal(size=csr[0].size - 1)
    db = torch.tensor(b, device=hip_device)
    for side in ("left", "right"):
        out = []
        for algo in ("levels", "single", "single"):
            g.set_solve_algorithm(algo)
            x = torch.zeros_like(db)
            getattr(g, f"solve_{side}")(db, x)
            out.append(x.cpu().numpy())
        assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2]), side
        if prec == "f64":
            ref = o.solve(side, b)
            assert np.linalg.norm(out[0] - ref) <= 1e-12 * np.linalg.norm(ref), side


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("shape,rows_per_level", [
    ((2000, 801, 4, 3, 32), (1, 128)),      # three waves per CU
    ((1500, 601, 4, 3, 1), (128, 384)),     # four
    ((4000, 1601, 4, 3, 1), (384, 4000)),   # rows walked one group after the other
    ((20000, 8003, 4, 3, 4), (384, 4000)),
])
def test_single_launch_forms_equal_levels(hip_device, shape, rows_per_level, prec):
    """The forms of the single-launch solve, chosen by block rows per level (of
    256 CUs), and the product folded into them: the level launches' bits."""
    import torch
    csr, piv, bs = _kkt(*shape)
    g = ca.BlockiLDLt(*csr, piv, bs, prec)
    g.compute(0, 1.0, 1e-4)
    lo, hi = rows_per_level
    assert lo < bs.size / (g.get_int("lvl_off").size - 1) <= hi
    A = ca.CSRMatrixSPMV(*csr)
    b = torch.tensor(np.random.default_rng(8).normal(size=csr[0].size - 1), device=hip_device)
    out = {}
    for algo in ("levels", "single"):
        g.set_solve_algorithm(algo)
        for op in ("left", "right", "product"):
            x = torch.zeros_like(b)
            if op == "product":
                assert g.left_product(A, b, x) == (algo == "single")
            else:
                getattr(g, f"solve_{op}")(b, x)
            out[algo, op] = x.cpu().numpy()
    for op in ("left", "right", "product"):
        assert np.array_equal(out["levels", op], out["single", op]), op


@pytest.mark.parametrize("algo,sweeps", [("levels", 0), ("single", 0), ("jacobi", 2)])
def test_iterates_do_not_depend_on_check_period(hip_device, algo, sweeps):
    import torch
    csr, piv, bs = _kkt(1500, 601, 4, 3, 16)
    g = ca.BlockiLDLt(*csr, piv, bs, "f64")
    g.compute(0, 1.0, 1e-4)
    g.set_solve_algorithm(algo, sweeps)
    A = ca.CSRMatrixSPMV(*csr)
    b = torch.tensor(np.random.default_rng(2).normal(size=csr[0].size - 1), device=hip_device)
    for max_it in (1, 2, 3, 5, 8):
        out = []
        for period in (1, 2, 3, 20):
            q = ca.SQMR(A, 1e-300, max_it, g, true_residual_period=period, max_restarts=0)
            x = torch.zeros_like(b)
            q.solve(b, x)
            assert q.result["iterations"] == max_it
            out.append(x.cpu().numpy())
        for x in out[1:]:
            assert np.array_equal(out[0], x), (max_it, algo)


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_nan_reaches_the_rows_of_the_substitution(hip_device, prec):
    """A NaN in a pivot block's U_ii reaches the solution's rows that back and
    forward substitution with U_ii give NaN (zeros beside it included) and no
    others, in every schedule; blocks beside the diagonal there are none."""
    import scipy.sparse as sp
    import torch
    rng = np.random.default_rng(11)
    hs = np.concatenate([np.arange(1, 33), [32, 17, 8]])
    bs = np.concatenate([[0], np.cumsum(hs)[:-1]]).astype(np.int32)
    blocks, bad = [], []
    for b, h in zip(bs, hs):
        a = np.triu(rng.normal(size=(h, h)) * (rng.random((h, h)) < 1.5 / h), 1)
        blocks.append(a + a.T + np.diag(rng.normal(size=h) + 3.0))
        bad.append(b + rng.integers(h))
    A = sp.block_diag(blocks).tocsr()
    A.sort_indices()
    n = A.shape[0]
    val = A.data.copy()
    rows = np.repeat(np.arange(n), np.diff(A.indptr))
    val[(rows == A.indices) & np.isin(rows, bad)] = np.nan
    csr = (A.indptr.astype(np.int32), A.indices.astype(np.int32), val)
    args = (*csr, np.arange(n, dtype=np.int32), bs)
    g = ca.BlockiLDLt(*args, prec)
    g.compute(0, 1.0, 1e-4)
    # U_ii as stored (dense, block after block)
    U = g.get_real("fval_store")
    b = rng.normal(size=n)
    ref = {"left": b.copy(), "right": b.copy()}
    for k, (f, h) in enumerate(zip(bs, hs)):
        u = U[(hs[:k] ** 2).sum():][:h * h].reshape(h, h).astype(np.float64)
        assert np.isnan(u[bad[k] - f]).all()
        inv = np.zeros((h, h))     # columns of the inverse by back substitution
        beside = (np.triu(u, 1) != 0).any()
        for c in range(h):
            for r in range(c, -1, -1):
                s = sum((u[r, j] * inv[j, c] for j in range(r + 1, c + 1)), 0.0)
                inv[r, c] = 1.0 / u[r, r] if r == c else -s / u[r, r] if beside else 0.0
        for side, m in (("left", inv.T), ("right", inv)):
            ref[side][f:f + h] = [sum(m[r, c] * b[f + c] for c in range(h) if m[r, c] != 0)
                                  for r in range(h)]
    db = torch.tensor(b, device=hip_device)
    for algo, sweeps in (("levels", 0), ("single", 0), ("jacobi", 1)):
        g.set_solve_algorithm(algo, sweeps)
        for side, want in ref.items():
            x = torch.zeros_like(db)
            getattr(g, f"solve_{side}")(db, x)
            x = x.cpu().numpy()
            assert np.array_equal(np.isnan(x), np.isnan(want)), (algo, side)
            ok = ~np.isnan(want)
            assert ok.any()
            assert np.linalg.norm((x - want)[ok]) <= \
                (1e-12 if prec == "f64" else 1e-5) * np.linalg.norm(want[ok]), (algo, side)
