"""The factor kernels at the sizes where their chunks, lists and masks end,
bit for bit against the oracle: pair lists over one chunk of 64, block rows
and columns of more blocks than one round of lanes, one-row blocks, 2x2
pivots that widen a block's row mask, dense-ish blocks beside one-entry ones,
levels of one block and of thousands."""
import numpy as np
import pytest

import culip_amd as ca
import oracle_lib as ol
from conftest import sym_problem

pytestmark = pytest.mark.gpu


def _compare(csr, piv, bs, prec="f64", pivoting="static", fill=0, ff=1.0, thr=1e-4):
    rp, ci, cv = csr
    g = ca.BlockiLDLt(rp, ci, cv, piv, bs, prec)
    g.set_pivoting(pivoting)
    g.compute(fill, ff, thr)
    o = ol.OracleBildlt(rp, ci, cv, piv, bs, "f" if prec == "f32" else "d")
    o.set_pivoting(pivoting)
    # the library's default arithmetic of an FP32 factor's 2x2 pivots
    o.set_pivot_precision("f64")
    o.symbolic(fill, ff)
    o.factor(thr)
    for nm in ("fblocks", "fix_store", "perm", "fis_piv"):
        assert np.array_equal(g.get_int(nm), o.get(nm)), nm
    for nm in ("fval_store", "tri", "row_norms"):
        assert np.array_equal(g.get_real(nm), o.get(nm)), nm


@pytest.mark.parametrize("n,m,o,c,B,order,prec,pivoting", [
    (2000, 800, 4, 3, 32, "color", "f64", "static"),
    (2600, 1001, 4, 3, 32, "natural", "f32", "static"),
    (2600, 1001, 4, 3, 32, "color", "f64", "rook"),
    (701, 280, 6, 4, 8, "natural", "f64", "static"),
    (1203, 481, 6, 4, 16, "color", "f32", "bk"),
    (4097, 1300, 4, 3, 1, "color", "f64", "static"),
    (9001, 3600, 6, 4, 8, "color", "f64", "static"),
    (20001, 7003, 4, 3, 31, "color", "f64", "static"),
])
def test_kkt_factor_equals_oracle(hip_device, n, m, o, c, B, order, prec, pivoting):
    k = ca.KKT(n, m, o, c, seed=n)
    p = ca.Prep(k.row_ptr, k.col, k.val, n, B,
                ca.ORDER_BLOCK_COLOR if order == "color" else ca.ORDER_NATURAL)
    _compare((p.row_ptr, p.col, p.val), p.piv_starts, p.block_starts, prec, pivoting)


@pytest.mark.parametrize("n_blocks,bmax,density,fill,ff,thr,prec", [
    (90, 12, 0.03, 0, 1.0, 1e-4, "f64"),     # more than 64 blocks in a column, 2x2 pivots
    (90, 12, 0.03, 0, 1.0, 1e-4, "f32"),
    (40, 32, 0.05, 1, 1.5, 1e-3, "f64"),     # lists beyond the small forms
    (70, 6, 0.1, 0, 4.0, 0.0, "f64"),
])
def test_two_by_two_factor_equals_oracle(hip_device, n_blocks, bmax, density, fill, ff, thr, prec):
    csr, piv, bs, _ = sym_problem(n_blocks=n_blocks, bmax=bmax, density=density, seed=n_blocks)
    _compare(csr, piv, bs, prec, fill=fill, ff=ff, thr=thr)


@pytest.mark.parametrize("n_blocks,bmax,density,prec,pivoting", [
    (200, 4, 0.03, "f64", "static"), (200, 4, 0.03, "f32", "static"),
    (150, 8, 0.02, "f64", "static"), (90, 12, 0.01, "f32", "static"), (90, 12, 0.01, "f64", "bk"),
])
def test_columns_beside_two_by_two_pivots_equal_oracle(hip_device, n_blocks, bmax, density, prec,
                                                       pivoting):
    """Blocks of one to four entries in a single column whose rows belong to
    2x2 pivots (most blocks of these sparse patterns)."""
    csr, piv, bs, _ = sym_problem(n_blocks=n_blocks, bmax=bmax, density=density, seed=7)
    _compare(csr, piv, bs, prec, pivoting=pivoting)
