"""The LDS tile kernel of the MFMA products at the edges of its tiles.

Sizes: 1473 x 1500 runs on the 64 x 64 tiles (partial last row and column of tiles), 523 x 540 on
the 32 x 32 tiles; K covers one element, partial and whole K stages of 16 and one element more.
Every storage order and type of the operands, against numpy.

Tolerance: an entry of a product of K terms in FP64 (fused multiply-adds in any order) is off by at
most (K + 2) eps times the sum of the absolute products; the three real products of the complex
form sum terms of (|Ar| + |Ai|)(|Br| + |Bi|) <= 2 |A||B| and combine three of them, so 8 (K + 4) eps
(|A| |B|) covers both.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


@pytest.fixture(scope="module")
def rt():
    from alf_amd import runtime
    runtime.load_library()
    return runtime


def operand(rng, rows, cols, op, cplx):
    shape = (rows, cols) if op == "N" else (cols, rows)
    a = rng.standard_normal(shape)
    return a + 1j * rng.standard_normal(shape) if cplx else a


def apply(op, a):
    return a if op == "N" else (a.T if op == "T" else a.conj().T)


@pytest.mark.parametrize("m,n", [(1473, 1500), (523, 540)])
@pytest.mark.parametrize("k", [1, 15, 16, 17, 47])
@pytest.mark.parametrize("opa,opb,ca,cb", [
    ("N", "N", False, True), ("N", "N", True, False), ("N", "N", True, True), ("C", "N", True, True),
    ("N", "C", True, True), ("C", "C", True, True), ("T", "T", True, True), ("T", "C", False, True),
    ("C", "T", True, False)])
def test_tile_edges(rt, m, n, k, opa, opb, ca, cb):
    rng = np.random.default_rng(1000 * k + m)
    a, b = operand(rng, m, k, opa, ca), operand(rng, k, n, opb, cb)
    got = rt.gemm(a, b, opa, opb)
    pa, pb = apply(opa, a), apply(opb, b)
    bound = 8 * (k + 4) * EPS * (np.abs(pa) @ np.abs(pb))
    assert (np.abs(got - pa @ pb) <= bound).all()


@pytest.mark.parametrize("m,n", [(1473, 1500), (523, 540)])
def test_tile_accumulates_with_alpha_and_beta(rt, m, n):
    rng = np.random.default_rng(m)
    k, alpha, beta = 33, 0.7 - 0.2j, -1.1 + 0.4j
    a, b = operand(rng, m, k, "N", True), operand(rng, k, n, "C", True)
    c = operand(rng, m, n, "N", True)
    got = rt.gemm(a, b, "N", "C", alpha=alpha, beta=beta, Cin=c)
    bound = 8 * (k + 8) * EPS * (abs(alpha) * (np.abs(a) @ np.abs(b).T) + abs(beta) * np.abs(c))
    assert (np.abs(got - (alpha * (a @ b.conj().T) + beta * c)) <= bound).all()
