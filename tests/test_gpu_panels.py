"""GPU parity of the panel kernels and the level solves at the sizes where their tiles end: two
cliques of w0 and w1 columns, each coupled to all s columns of a third, so that two fronts with s
rows below them are extended-added into a third. The matrices are 3 I plus a symmetric random part
of norm below 1.2 (condition below 3), so a backward-stable factor or solve of n <= 700 columns is
off by at most about n u times that: 3e-13 in FP64 (1e-12 asserted, the comparison being as inexact) and
1.7e-4 in FP32. Every side of a block
solve is the bits of the same side alone. The LDL^T solve's columns at its own limits (a panel of 64
columns, 1 024 rows in the small form of the backward pass) are the oracle's bits."""
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


def rel(a, b):
    return np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(np.asarray(b))


SHAPES = [(1, 2, 1), (15, 17, 16), (16, 31, 33), (63, 65, 15), (64, 66, 64), (127, 129, 17), (128, 130, 63),
          (200, 96, 129), (257, 191, 65), (300, 130, 200)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("precision", ["fp64", "fp32", "mixed"])
def test_fronts_with_rows_below(gpu, shape, precision):
    a = cliques(*shape)
    n, ptr, idx, val = dense_to_csr(a)
    print(f"panels {shape} {precision}", flush=True)
    up = upper(n, ptr, idx, val)
    f = CH.Factor(CH.Symbolic(CH.UpperColumns(n, *up)), up[2], precision=precision)
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


@pytest.mark.parametrize("shape", [(15, 17, 16), (128, 130, 63), (300, 130, 200)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nrhs", [15, 16, 17, 32, 33])
def test_block_solves_are_the_bits_of_lone_ones(gpu, shape, precision, nrhs):
    n, ptr, idx, val = dense_to_csr(cliques(*shape))
    up = upper(n, ptr, idx, val)
    f = CH.Factor(CH.Symbolic(CH.UpperColumns(n, *up)), up[2], precision=precision)
    bs = [np.cos(np.arange(n) * (0.1 + 0.01 * k)) for k in range(nrhs)]
    for x, b in zip(f.solve_many(bs), bs):
        assert np.array_equal(x, f.solve(b))


@pytest.mark.parametrize("shape", [(1, 2, 1), (63, 65, 64), (64, 129, 66), (3, 200, 130), (2, 40, 990), (2, 40, 1030)],
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
