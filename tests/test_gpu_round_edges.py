"""Metropolis rounds and passes where their own state reaches the end of its range, against the oracle's
sequential visits.

Tolerances: the fields and the random-stream position are the oracle's; G and PHASE to 1e-10, as in
the other comparisons of whole sweeps (different summation orders in FP64).
"""
import cmath
import math

import numpy as np
import pytest

from helpers import fields_for, hubbard, oracle, rel
from oracle.dqmc_oracle import gama, phi

pytestmark = pytest.mark.gpu

TOL = 1e-10


@pytest.fixture(scope="module")
def rt():
    from alf_amd import runtime
    runtime.load_library()
    return runtime


def recorded(s):
    """Per slice of the oracle's sweeps, the weights |ratio| of its accepted flips."""
    slices, inner = [], s.upgrade2

    def upgrade2(G, n, nt, new):
        P, typ, g, E, alpha = s.m.scalars[n]
        old, g_pp = int(s.f[n, nt]), complex(G[P, P])
        toggle = inner(G, n, nt, new)
        if toggle:
            z1 = g * (phi(new, typ) - phi(old, typ))
            e = cmath.exp(z1 * E)
            ratio = (e - (e - 1.0) * g_pp) * cmath.exp(z1 * alpha)
            slices[-1].append(abs(ratio) ** s.m.n_sun * gama(new, typ) / gama(old, typ))
        return toggle

    def slice_of(call):
        def wrap(G, nt):
            slices.append([])
            return call(G, nt)
        return wrap

    s.upgrade2, s.wrapgrup, s.wrapgrdo = upgrade2, slice_of(s.wrapgrup), slice_of(s.wrapgrdo)
    return slices


@pytest.mark.parametrize("n_sun,shift", [(1, 40.0), (2, 20.0), (3, 15.0), (4, 12.0), (5, 9.0)])
def test_weights_of_a_block_beyond_the_range_of_a_double(rt, n_sun, shift):
    """A field that couples to a large real shift of the operator: every flip towards the favoured
    value is taken, with a weight of up to 1e80, so the product of the flips of one block (up to 16
    of them) is far beyond the largest double while each weight is inside it."""
    ham = hubbard(L1=5, L2=4, beta=0.6, nwrap=3, U=4.0)
    ham.N_SUN = n_sun
    for o in ham.Op_V:
        o.alpha = 1j * shift
    f = fields_for(ham, 3)
    u = np.random.default_rng(7).random(2 * 3 * len(ham.Op_V) * ham.Ltrot + 1)
    s = oracle(ham, f, u)
    slices = recorded(s)
    e = rt.Engine(ham)
    e.set_fields(f)
    e.set_tape(u)
    s.init()
    e.init()
    s.sweep()
    e.sweep(1)
    assert max(sum(math.log10(r) for r in x[:16]) for x in slices) > 320
    assert max(r for x in slices for r in x) < 1e150
    assert np.array_equal(e.get_fields(), s.f)
    assert e.rng_position() == s.rng.pos
    assert rel(e.get_green(), s.G) < TOL
    assert abs(e.get_phase() - s.phase) < TOL
    e.close()


@pytest.mark.parametrize("ltrot", [1, 2, 3, 4, 5, 7])
def test_windows_of_visits(rt, ltrot):
    """The visits of a pass are prepared half of its slices at a time: passes of one window and of
    several with and without a remainder, from a tape and from the Philox stream, which a delay
    beyond the block kernel's reads in windows of uniforms and must follow to the same fields."""
    ham = hubbard(L1=3, L2=4, beta=0.1 * ltrot, nwrap=2, U=4.0)
    f = fields_for(ham, 4)
    u = np.random.default_rng(9).random(2 * 2 * 3 * len(ham.Op_V) * ltrot)
    s = oracle(ham, f, u)
    s.init()
    e = rt.Engine(ham, delay=8)
    e.set_fields(f)
    e.set_tape(u)
    e.init()
    for _ in range(2):
        s.sweep()
        e.sweep(1)
        assert np.array_equal(e.get_fields(), s.f) and e.rng_position() == s.rng.pos
        assert rel(e.get_green(), s.G) < TOL
    e.close()
    got = []
    for delay in (8, 40):
        e = rt.Engine(ham, delay=delay)
        e.set_fields(f)
        e.set_philox(21, 2)
        e.init()
        e.sweep(4)
        got.append((e.get_fields(), e.rng_position(), e.get_green()))
        e.close()
    assert np.array_equal(got[0][0], got[1][0]) and got[0][1] == got[1][1] == 4 * 2 * 3 * len(ham.Op_V) * ltrot
    assert rel(got[1][2], got[0][2]) < TOL


@pytest.mark.parametrize("delay,n_sun", [(1, 2), (15, 1), (16, 2), (17, 3), (31, 2), (32, 2), (32, 4), (32, 5)])
def test_rounds_of_single_operator_sites(rt, delay, n_sun):
    """One operator per site on a lattice of several blocks: rounds that fill up, flips carried from
    block to block of a round, blocks cut short by their 16th flip, and (after a first sweep that
    accepts little) slices that outgrow the rounds planned for them."""
    ham = hubbard(L1=7, L2=14, beta=0.6, nwrap=3, U=0.6)
    ham.N_SUN = n_sun
    f = fields_for(ham, 3)
    per = 2 * 3 * ham.Ltrot * len(ham.Op_V)
    u = np.random.default_rng(7).random(3 * per).reshape(-1, 3)
    u[:per // 3, 2] = 1.0 - 2.0**-40      # the decisions' numbers
    u[per // 3:, 2] *= 0.2
    u = u.ravel()
    s = oracle(ham, f, u)
    slices = recorded(s)
    e = rt.Engine(ham, delay=delay)
    e.set_fields(f)
    e.set_tape(u)
    s.init()
    e.init()
    most = []
    for _ in range(3):
        del slices[:]
        s.sweep()
        e.sweep(1)
        most.append(max(len(x) for x in slices))
        assert np.array_equal(e.get_fields(), s.f)
        assert rel(e.get_green(), s.G) < TOL
        assert abs(e.get_phase() - s.phase) < TOL
        assert e.rng_position() == s.rng.pos
    # the largest slice of the first sweep plans the rounds of the second
    assert min(most) > max(delay, 16) and most[1] > -(-most[0] // delay) * delay
    c = e.control()
    assert c["NC_up"] == s.ctrl.NC_up and c["ACC_up"] == s.ctrl.ACC_up
    e.close()


@pytest.mark.parametrize("L1,L2,chains,fusion", [(16, 16, 16, False), (7, 9, 256, True), (17, 16, 12, True)])
def test_flush_of_a_batch(rt, L1, L2, chains, fusion):
    """Batches whose 64 x 64 tiles fill the device (16 tiles a chain, one with a remainder, 25 with
    remainders): the rounds' factors and the batched flush, against the same chains one at a time."""
    ham = hubbard(L1=L1, L2=L2, beta=0.4, nwrap=2)
    fs = [fields_for(ham, 20 + z) for z in range(chains)]
    b = rt.BatchEngine([ham] * chains)
    b.round_fusion(fusion)
    for z in range(chains):
        b.chain(z).set_fields(fs[z])
        b.set_philox(31, z)
    b.init()
    b.sweep(2)
    for z in (0, chains // 2, chains - 1):
        e = rt.Engine(ham)
        e.set_fields(fs[z])
        e.set_philox(31, z)
        e.init()
        e.sweep(2)
        b.chain(z)
        assert np.array_equal(b.get_fields(), e.get_fields()) and not np.array_equal(e.get_fields(), fs[z])
        assert rel(b.get_green(), e.get_green()) < TOL
        assert abs(b.get_phase() - e.get_phase()) < TOL
        e.close()
    b.close()
