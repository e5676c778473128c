"""Metropolis rounds at the edges of their blocks: depths around the 16-acceptance blocks and the
32-row tables, several operators of both types on one site, numbers of colours on both sides of
the per-visit renormalisation, and slices that outgrow their planned rounds, against the oracle's
sequential visits.

Tolerances: the fields, counters and random-stream positions are the oracle's; G and PHASE to
1e-10, as in the other comparisons of whole sweeps (different summation orders in FP64).
"""
import copy

import numpy as np
import pytest

from helpers import fields_for, hubbard, oracle, rel

pytestmark = pytest.mark.gpu

TOL = 1e-10


@pytest.fixture(scope="module")
def rt():
    from alf_amd import runtime
    runtime.load_library()
    return runtime


def model(n_sun, ops):
    ham = hubbard(L1=5, L2=4, beta=0.6, nwrap=3, U=0.6)
    ham.N_SUN = n_sun
    f = fields_for(ham, 3)
    if ops == "several":
        # every site again with a two-valued field, every third one a third time
        second = [copy.copy(o) for o in ham.Op_V]
        for o in second:
            o.type = 1
        third = [copy.copy(o) for o in ham.Op_V[::3]]
        r = np.random.default_rng(5)
        f = np.concatenate([f, 2 * r.integers(0, 2, f.shape) - 1, f[::3]]).astype(f.dtype)
        ham.Op_V = ham.Op_V + second + third
        ham.nsigma = type(ham.nsigma).make(len(ham.Op_V), ham.Ltrot)
        ham.nsigma.t[:] = [o.type for o in ham.Op_V]
        ham.nsigma.f[:, :] = f
    return ham, f


@pytest.mark.parametrize("ops", ["one", "several"])
@pytest.mark.parametrize("delay,n_sun", [(1, 2), (15, 1), (16, 2), (17, 3), (31, 2), (32, 2), (32, 4), (32, 5)])
def test_rounds_follow_sequential_visits(rt, delay, n_sun, ops):
    ham, f = model(n_sun, ops)
    per = 2 * ham.Ltrot * int(np.sum([3 if o.type == 2 else 2 for o in ham.Op_V]))
    # the first sweep accepts little, so the rounds planned for the second one are too few
    u = np.concatenate([np.full(per, 1.0 - 2.0**-40), np.random.default_rng(7).random(2 * per)])
    s = oracle(ham, f, u)
    e = rt.Engine(ham, delay=delay)
    e.set_fields(f)
    e.set_tape(u)
    s.init()
    e.init()
    for _ in range(3):
        s.sweep()
        e.sweep(1)
        assert np.array_equal(e.get_fields(), s.f)
        assert rel(e.get_green(), s.G) < TOL
        assert abs(e.get_phase() - s.phase) < TOL
        assert e.rng_position() == s.rng.pos
    c = e.control()
    assert c["NC_up"] == s.ctrl.NC_up and c["ACC_up"] == s.ctrl.ACC_up
    assert c["ACC_up"] > 0.2 * c["NC_up"]
    e.close()


@pytest.mark.parametrize("L1,L2,delay", [(5, 4, 1), (5, 4, 15), (3, 11, 16), (7, 5, 17), (4, 12, 32)])
def test_flush_of_a_round_in_one_launch_and_in_two(rt, L1, L2, delay):
    """G after the slices of one interval with the factors X and Y of each round formed inside the
    flush and by a kernel of their own: the same sums in another order, so 1e-12 of G.  (Depths
    below, at and above 16 columns, Ndim with and without a remainder of 16.)"""
    ham = hubbard(L1=L1, L2=L2, beta=0.6, nwrap=3, U=2.0)
    f = fields_for(ham, 3)
    got = []
    for on in (1, 0):
        e = rt.Engine(ham, delay=delay)
        e.round_fusion(bool(on))
        e.set_fields(f)
        e.set_philox(11, 0)
        e.init()
        for nt in range(3):
            e.wrapgrup(nt, e.get_phase())
        got.append((e.get_green(), e.get_fields(), e.rng_position()))
        e.close()
    assert np.array_equal(got[0][1], got[1][1]) and got[0][2] == got[1][2]
    assert not np.array_equal(got[0][1], f)
    assert rel(got[1][0], got[0][0]) < 1e-12
