"""Rounding errors of a front's first panel on the GPU, against residuals in 80-bit arithmetic.

With u the unit roundoff of the storage, pw the panel's columns, L11 its diagonal block and x a row
below it solved from b:

  * the root of a pivot is the correctly rounded square root: a diagonal matrix's factor is its
    entries' square roots;
  * an entry of L11 takes at most 7 subtractions of earlier blocks' products, 15 updates inside its
    block of 16 columns and a quotient, each a rounding (0.29 u rms) of at most (|L| |L|^T)_ij, which
    keeps the rms of (A - L L^T)_ij / (|L| |L|^T)_ij below sqrt(23) 0.29 u < 1.4 u;
  * an entry of x takes three roundings of its own size (b less the earlier products, the residual or
    quotient, the correction; 0.5 u together), the sums' own roundings being of products' size: the
    residual of a row is below u |x| |L11| / sqrt(pw) in the rms over the rows, |L11| being
    sqrt(pw) times its diagonal's size.

Sums carried on the running value instead (a rounding of it for each of 112 products) are three times
the last two bounds.
"""
import numpy as np
import pytest

from fieldcraft_amd import cholesky as CH

from matrices import dense_to_csr, upper

pytestmark = pytest.mark.gpu

UNIT = {"fp64": 2.0 ** -53, "fp32": 2.0 ** -24, "mixed": 2.0 ** -24}


def spd(n, seed):
    g = np.random.default_rng(seed).uniform(-1.0, 1.0, (n, n)) / np.sqrt(n)
    return (g + g.T) / np.sqrt(2.0) + 3.0 * np.eye(n)


def small_front(w, rows=100):
    """Three cliques of w columns, each coupled to a part of its own of the blocks above them: every one's
    front keeps its w columns with rows below."""
    sizes = np.cumsum([0, w, w, rows, w, rows + 50])
    a, b, s, c, t = (np.arange(sizes[k], sizes[k + 1]) for k in range(5))
    m = np.zeros((sizes[-1],) * 2, bool)
    for i, j in [(a, a), (b, b), (s, s), (c, c), (t, t), (a, s[:2 * rows // 3]), (b, s[rows // 3:]), (a, t[:rows // 2]),
                 (s, t[:rows]), (c, t[rows // 3:])]:
        m[np.ix_(i, j)] = m[np.ix_(j, i)] = True
    return np.where(m, spd(sizes[-1], w), 0.0)


def first_panel(a, precision):
    """The first supernode's columns of the factor and of the matrix (rounded to the storage)."""
    n, ptr, idx, val = dense_to_csr(a)
    up = upper(n, ptr, idx, val)
    sym = CH.Symbolic(CH.UpperColumns(n, *up))
    e = sym.export()
    rows, w = e["rows"][: e["rptr"][1]], int(e["first"][1])
    v, m = CH.Factor(sym, up[2], precision=precision).values(), len(rows)
    low = np.zeros((m, w))
    at = 0
    for c in range(w):
        low[c:, c] = v[at: at + m - c]
        at += m - c
    if precision != "fp64":
        a = a.astype(np.float32).astype(np.float64)
    return low, a[np.ix_(e["perm"][rows], e["perm"][rows[:w]])], sym


def check(low, a, u):
    pw = min(low.shape[1], 128)
    low, a = low[:, :pw].astype(np.longdouble), a[:, :pw]
    r = np.abs(a - low @ low[:pw].T).astype(np.float64) / u
    tri = np.tril_indices(pw)
    diag = np.sqrt(np.mean((r[tri] / (np.abs(low) @ np.abs(low[:pw]).T)[tri].astype(np.float64)) ** 2))
    below, x, l11 = r[pw:], low[pw:].astype(np.float64), low[:pw].astype(np.float64)
    rows = np.sqrt(np.mean((np.linalg.norm(below, axis=1) / np.linalg.norm(x, axis=1) / np.linalg.norm(l11)) ** 2))
    print(f"diagonal block {diag:.3f} u, rows below {rows * np.sqrt(pw):.3f} u / sqrt({pw})", flush=True)
    assert diag <= 1.4
    assert rows <= 1.0 / np.sqrt(pw)


@pytest.mark.parametrize("w", [17, 33, 48, 64])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_a_small_fronts_rows(gpu, w, precision):
    print(f"small front {w} {precision}", flush=True)
    low, a, sym = first_panel(small_front(w), precision)
    assert sym.info()["kind_flops"]["small"] > 0 and low.shape[1] == w and low.shape[0] > w + 50
    check(low, a, UNIT[precision])


@pytest.mark.parametrize("n", [145, 200, 333])
@pytest.mark.parametrize("precision", ["fp64", "fp32", "mixed"])
def test_a_panels_rows(gpu, n, precision):
    print(f"panel {n} {precision}", flush=True)
    low, a, _ = first_panel(spd(n, n), precision)
    assert low.shape == (n, n)
    check(low, a, UNIT[precision])


def test_pivot_roots_are_correctly_rounded(gpu):
    d = np.exp2(np.random.default_rng(5).uniform(-600.0, 600.0, 4000))
    n, ptr, idx, val = len(d), np.arange(len(d) + 1), np.arange(len(d)), d
    sym = CH.Symbolic(CH.UpperColumns(n, ptr, idx, val))
    assert np.array_equal(CH.Factor(sym, val).values(), np.sqrt(d[sym.export()["perm"]]))
