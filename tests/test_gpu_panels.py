"""GPU parity of the panel kernels and the level solves at the sizes where their tiles end.

`cliques`: two blocks of w0 and w1 columns, each coupled to all s columns of a third. The analysis
merges one of the two with the s columns at no fill, so the factor has two fronts: w0 columns with
s rows below, and the rest.

`tree`: blocks of wa, wb, s, wb and t columns, A and B below S, S and C below T, each coupled to a part
of its own of the block above (A to some of T too), so that none merges for free: fronts of every
width with rows below, two children's columns on one of the parent's, several fronts in a level, and
children's entries in the update matrices. What the analysis made of it is asserted.

The matrices are 3 I plus a symmetric random part of norm below 1.2 (condition below 3), so a
backward-stable factor or solve of n <= 1 206 columns is off by at most about n u times that: 4e-13 in
FP64 (1e-12 asserted, the comparison being as inexact) and, the larger ones' condition being below 2.2,
1.7e-4 in FP32. Every side of a block solve is the bits of the same side alone. The LDL^T solve's columns at its own limits (a panel of 64
columns, the 1 152 entries of a column held ahead in the backward pass) are the oracle's bits."""
import numpy as np
import pytest

from fieldcraft_amd import cholesky as CH
from oracle import oracle as O

from matrices import dense_to_csr, upper

pytestmark = pytest.mark.gpu


def cliques(w0, w1, s, shift=3.0):
    n = w0 + w1 + s
    g = np.random.default_rng(1000 * w0 + 10 * w1 + s).uniform(-1.0, 1.0, (n, n)) / np.sqrt(n)
    a = (g + g.T) / np.sqrt(2.0)
    a[:w0, w0:w0 + w1] = 0.0
    a[w0:w0 + w1, :w0] = 0.0
    return a + shift * np.eye(n)


def tree(wa, wb, s, t):
    o = np.cumsum([0, wa, wb, s, wb, t])
    n = o[-1]
    A, B, S, C, T = (np.arange(o[k], o[k + 1]) for k in range(5))
    m = np.zeros((n, n), bool)
    q = 8 if wa < 40 else 3  # (a narrow front with many rows below would be merged into its parent)
    for i, j in [(A, A), (B, B), (S, S), (C, C), (T, T), (A, S[:2 * s // q]), (B, S[s // q:4 * s // q]), (A, T[:t // q]),
                 (S, T[:2 * t // 3]), (C, T[t // 3:t if q == 3 else t // 2])]:
        m[np.ix_(i, j)] = m[np.ix_(j, i)] = True
    g = np.random.default_rng(1000 * wa + wb).uniform(-1.0, 1.0, (n, n)) / np.sqrt(n)
    return np.where(m, (g + g.T) / np.sqrt(2.0), 0.0) + 3.0 * np.eye(n)


def rel(a, b):
    return np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(np.asarray(b))


SHAPES = [(1, 2, 1), (15, 17, 16), (16, 31, 33), (63, 65, 15), (64, 66, 64), (127, 129, 17), (128, 130, 63),
          (200, 96, 129), (257, 191, 65), (300, 130, 200)]


# the last: fronts of 33 and 40 columns with 130 to 600 rows below
TREES = [(15, 17, 80, 130), (16, 31, 65, 120), (63, 65, 64, 129), (64, 66, 100, 130),
         (127, 129, 97, 150), (128, 130, 129, 128), (200, 96, 129, 257), (257, 191, 129, 150), (40, 33, 200, 900)]


def check_factor(a, precision, sym, up, csr):
    n, ptr, idx, val = csr
    f = CH.Factor(sym, up[2], precision=precision)
    rounded = val if precision == "fp64" else val.astype(np.float32).astype(np.float64)
    ref = O.Factor(n, *upper(n, ptr, idx, rounded))
    assert rel(f.values(), ref.values()) <= {"fp64": 1e-12, "fp32": 1.7e-4, "mixed": 1.7e-4}[precision]
    b = np.sin(np.arange(n) * 0.9)
    if precision == "fp64":
        assert rel(f.solve(b), np.linalg.solve(a, b)) <= 1e-12
    else:
        x, rep = f.solve_refined(CH.Matrix(n, ptr, idx, val), b, target_berr=1e-12)
        assert rep["converged"], rep
        assert rel(x, np.linalg.solve(a, b)) <= 1e-10


@pytest.mark.parametrize("shape", TREES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("precision", ["fp64", "fp32", "mixed"])
def test_trees_of_fronts(gpu, shape, precision):
    a = tree(*shape)
    csr = dense_to_csr(a)
    up = upper(*csr)
    sym = CH.Symbolic(CH.UpperColumns(csr[0], *up))
    info, e = sym.info(), sym.export()
    print(f"tree {shape} {precision}", flush=True)
    assert info["fronts"] >= 4 and info["levels"] == 3
    assert info["kind_entries"]["extend_l"] > 0 and info["kind_entries"]["extend_u"] > 0
    w, m = np.diff(e["first"]), np.diff(e["rptr"])
    assert w[0] == shape[1] and m[0] - w[0] >= (512 if shape[3] == 900 else 16)
    check_factor(a, precision, sym, up, csr)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("precision", ["fp64", "fp32", "mixed"])
def test_fronts_with_rows_below(gpu, shape, precision):
    a = cliques(*shape)
    n, ptr, idx, val = dense_to_csr(a)
    print(f"panels {shape} {precision}", flush=True)
    up = upper(n, ptr, idx, val)
    check_factor(a, precision, CH.Symbolic(CH.UpperColumns(n, *up)), up, (n, ptr, idx, val))


@pytest.mark.parametrize("shape", [(15, 17, 16), (128, 130, 63), (300, 130, 200), (63, 65, 64, 129), (40, 33, 200, 900)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nrhs", [15, 16, 17, 32, 33])
def test_block_solves_are_the_bits_of_lone_ones(gpu, shape, precision, nrhs):
    n, ptr, idx, val = dense_to_csr((cliques if len(shape) == 3 else tree)(*shape))
    up = upper(n, ptr, idx, val)
    f = CH.Factor(CH.Symbolic(CH.UpperColumns(n, *up)), up[2], precision=precision)
    bs = [np.cos(np.arange(n) * (0.1 + 0.01 * k)) for k in range(nrhs)]
    for x, b in zip(f.solve_many(bs), bs):
        assert np.array_equal(x, f.solve(b))


@pytest.mark.parametrize("shape", [(1, 2, 1), (63, 65, 64), (64, 129, 66), (3, 200, 130), (2, 40, 990), (2, 40, 1030),
                                   (2, 40, 1160)],
                         ids=lambda s: "x".join(map(str, s)))
def test_ldlt_columns_are_the_oracles_bits(gpu, shape):
    a = cliques(*shape, shift=0.1)  # indefinite: 2 x 2 pivots
    n, ptr, idx, val = dense_to_csr(a)
    print(f"LDL^T {shape}", flush=True)
    up = O.from_symmetric(n, ptr, idx, val)
    f, ref = CH.LdltFactor(CH.Symbolic(CH.UpperColumns(n, *up)), up[2]), O.LdltFactor(n, *up)
    assert np.array_equal(f.values(), ref.values())
    b = np.sin(np.arange(n) * 0.9)
    assert np.array_equal(f.solve(b), ref.solve(b))
