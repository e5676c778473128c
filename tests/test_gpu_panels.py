"""The panels of the blocked QR at the edges of their kernels: rows at, below and above those that
1, 2, 4, 8, .. rows per lane hold, and panel widths 32, 16 and 4 with and without a remainder, in
the UDV decomposition of a product of slices against the oracle's.

Tolerance: Householder QR leaves errors of order n eps in Q's orthogonality and of n eps |A| in
Q R; 20 n eps of the largest entry covers the constant and the second decomposition.
"""
import numpy as np
import pytest

from helpers import fields_for, hubbard, oracle, rel
from oracle import dqmc_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L1,L2", [
    (4, 4), (4, 8), (3, 11), (8, 8), (5, 13), (8, 16), (3, 43), (16, 16),   # one lane's 1, 2, 4, 8 rows
    (3, 86), (16, 18), (16, 24), (5, 77), (16, 32),                         # width 32, 257 to 512 rows
    (19, 27), (24, 32), (25, 31), (32, 32),                                 # width 16, 513 to 1024 rows
    (25, 42),                                                               # width 4
])
def test_decomposition_at_the_edges_of_the_panels(L1, L2):
    from alf_amd import runtime as rt
    ham = hubbard(L1=L1, L2=L2, beta=0.4, nwrap=2)
    f = fields_for(ham, 2)
    n = ham.Ndim
    s = oracle(ham, f, np.zeros(1), presort=True)
    e = rt.Engine(ham)
    e.set_fields(f)
    e.udv_reset(rt.ALFQ_UDVR, "R")
    e.wrapur(0, 2)
    e.wrapur(2, 4)
    U, D, V = e.get_udv(rt.ALFQ_UDVR)
    e.close()
    uo = s.wrapur(2, 4, s.wrapur(0, 2, O.UDV.identity(n, "R")))
    tol = 20 * n * np.finfo(float).eps
    assert np.abs(U.conj().T @ U - np.eye(n)).max() < tol
    assert rel((U * D) @ V, (uo.U * uo.D) @ uo.V) < tol
    assert rel(np.sort(D.real), np.sort(uo.D.real)) < tol
