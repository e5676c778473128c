"""The LDS tile kernel of the MFMA products over several K stages, and with gathered and scaled operands.

Sizes: 507 x 510 keeps the 32 x 32 tiles for every K here (partial last row and column of tiles), from a
part of one stage of 16 to whole stages with one element more; tests/test_gemm_rule_host.py checks which
kernel these sizes take.  The batches run the hopping wraps, the UDV chain, QR and CGR on the tiles: Ndim
99 on 32 x 32 and 125 on 64 x 64, both with a partial last K stage, against the same chains one at a time,
which run on the direct kernel.

Tolerances: an entry of a product of K terms in FP64 (fused multiply-adds in any order) is off by at most
(K + 2) eps times the sum of the absolute products; the three real products of the complex form sum terms
of (|Ar| + |Ai|)(|Br| + |Bi|) <= 2 |A||B| and combine three of them, so 8 (K + 4) eps (|A| |B|) covers
both.  Trajectories of the batches to 1e-10 as in the other comparisons of whole sweeps.  One slice with
FP32 wraps: two products of K = Ndim terms with row sums of |exp(-dtau T)| below 1.5 on each of the two
sides, 2 x 2 x 1.5^2 (K + 2) eps32 = 7e-5 of G, and the flips of the slice amplify it by a few: 1e-3.
"""
import numpy as np
import pytest

from helpers import fields_for, hubbard, rel

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


@pytest.mark.parametrize("k", [15, 16, 17, 33, 47])
@pytest.mark.parametrize("opa,opb,ca,cb", [
    ("N", "N", False, True), ("N", "N", True, False), ("N", "N", True, True), ("C", "N", True, True),
    ("N", "C", True, True), ("C", "C", True, True), ("T", "T", True, True), ("T", "C", False, True),
    ("C", "T", True, False)])
def test_stages_of_the_small_tile(rt, k, opa, opb, ca, cb):
    rng = np.random.default_rng(100 * k)
    a, b = operand(rng, 507, k, opa, ca), operand(rng, k, 510, opb, cb)
    alpha, beta = 0.7 - 0.2j, -1.1 + 0.4j
    c = operand(rng, 507, 510, "N", True)
    pa, pb = apply(opa, a), apply(opb, b)
    mag = np.abs(pa) @ np.abs(pb)
    assert (np.abs(rt.gemm(a, b, opa, opb) - pa @ pb) <= 8 * (k + 4) * EPS * mag).all()
    got = rt.gemm(a, b, opa, opb, alpha=alpha, beta=beta, Cin=c)
    bound = 8 * (k + 8) * EPS * (abs(alpha) * mag + abs(beta) * np.abs(c))
    assert (np.abs(got - (alpha * (pa @ pb) + beta * c)) <= bound).all()


@pytest.mark.parametrize("L1,L2,chains", [(9, 11, 32), (5, 25, 128)])
def test_scaled_and_gathered_operands(rt, L1, L2, chains):
    ham = hubbard(L1=L1, L2=L2, beta=0.4, nwrap=2)
    fs = [fields_for(ham, 40 + z) for z in range(chains)]
    b = rt.BatchEngine([ham] * chains)
    for z in range(chains):
        b.chain(z).set_fields(fs[z])
        b.set_philox(13, z)
    b.init()
    b.sweep(2)
    for z in (0, chains // 3, chains - 1):
        e = rt.Engine(ham)
        e.set_fields(fs[z])
        e.set_philox(13, z)
        e.init()
        e.sweep(2)
        b.chain(z)
        assert np.array_equal(b.get_fields(), e.get_fields())
        assert rel(b.get_green(), e.get_green()) < 1e-10
        assert abs(b.get_phase() - e.get_phase()) < 1e-10
        e.close()
    b.close()


@pytest.mark.parametrize("L1,L2,chains", [(9, 11, 32), (5, 25, 128)])
def test_fp32_wraps_with_a_partial_stage(rt, L1, L2, chains):
    ham = hubbard(L1=L1, L2=L2, beta=0.4, nwrap=2)
    fs = [fields_for(ham, 70 + z) for z in range(chains)]

    def slices(eng, z):
        """G and the fields after a slice up and after the one down again (chain z of eng)."""
        out = []
        for call, nt in ((eng.wrapgrup, 0), (eng.wrapgrdo, 1)):
            call(nt)
            if eng is b:
                eng.chain(z)
            out.append((eng.get_green(), eng.get_fields()))
        return out

    b = rt.BatchEngine([ham] * chains)
    b.set_precision(rt.PREC_FP32_WRAPS)
    for z in range(chains):
        b.chain(z).set_fields(fs[z])
        b.set_philox(13, z)
    b.init()
    z = chains - 1
    e = rt.Engine(ham)
    e.set_precision(rt.PREC_FP32_WRAPS)
    e.set_fields(fs[z])
    e.set_philox(13, z)
    e.init()
    exact = rt.Engine(ham)
    exact.set_fields(fs[z])
    exact.set_philox(13, z)
    exact.init()
    for (gb, fb), (ge, fe), (gx, _) in zip(slices(b, z), slices(e, z), slices(exact, z)):
        assert np.array_equal(fb, fe)
        assert rel(gb, ge) < 1e-3
        assert rel(gb, gx) > 1e-9       # FP32 arithmetic did run
    for x in (b, e, exact):
        x.close()
