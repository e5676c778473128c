"""Device memory of one chain (alfq_chain_bytes): what is kept for the Metropolis visits of a pass must
not make a chain larger than the uniforms of a sweep did (8 bytes for each of 2 or 3 numbers a visit,
two passes), so that batches and serving lanes of the same size still fit.  The limits are the bytes of
a chain in that form."""
import pytest

from helpers import hubbard


@pytest.mark.parametrize("L1,L2,beta,kind,limit", [
    (4, 4, 5.0, 2, 1933312), (16, 16, 10.0, 2, 55615488), (16, 16, 10.0, 1, 55205888), (5, 5, 4.5, 1, 2215936),
    (12, 24, 12.0, 2, 75042816), (24, 24, 4.0, 2, 201695232)])
def test_a_chain_is_no_larger(L1, L2, beta, kind, limit):
    from alf_amd import runtime as rt
    ham = hubbard(L1=L1, L2=L2, beta=beta, nwrap=10)
    for o in ham.Op_V:
        o.type = kind
    assert rt.chain_bytes(ham) <= limit
