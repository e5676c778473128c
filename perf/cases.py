"""The work that users of the sweep engine have it do, as cases that can be timed and compared.

A case is one way of driving the engine, through ``alf_amd.runtime`` only:

* ``chain``    one Markov chain, whole sweeps (replayed graphs), G and the fields read back
* ``bin``      the same with the equal-time (and time-displaced) measurements: sweeps of a bin,
               then the bin's sums
* ``batch``    many chains in one context, every launch covering all of them
* ``segment``  a host that drives the slices itself, as the Fortran host does: up through one
               stabilisation interval (WRAPGRUP, WRAPUR, CGR) and down again (WRAPGRDO, WRAPUL,
               CGR), each call returning before the next is made
* ``init``     a new configuration of fields: the left chain of UDV states and G at tau = 0

Sizes are those of the benchmark, the tests and the serving stream: square lattices of 4 x 4 to
32 x 32, the honeycomb with a flux (complex hopping), dense and checkerboard hopping, FP64 and
the int8 split products, chains of one and of uneven inverse temperature.  Fields are uniform
four-state from the seed and the random stream is Philox with the seed as its key.
"""
from __future__ import annotations

import math
from functools import lru_cache

import numpy as np

from alf_amd.host.hamiltonian import HubbardParams, hubbard_ham_set
from alf_amd.runtime import ALFQ_UDVL, ALFQ_UDVR, PREC_INT8_SPLIT, BatchEngine, Engine

FIELD_VALUES = np.array([-2, -1, 1, 2], dtype=np.int64)
# sweeps before a pass: the eager one, the capture of both buffer parities, and for one chain a
# few more, in which the number of delayed-update rounds per slice (and with it the graph) settles
WARM = {"chain": 6, "bin": 6, "batch": 3}


def listed():
    """The cases that are timed each time."""
    base = {"lattice": "Square", "u": 4.0, "nwrap": 10, "flux": 0, "checkerboard": False, "chains": 1,
            "split": False, "tau": False, "beta_min": 0.0, "sweeps": 1}
    rows = [
        # the smallest whole call: the 4 x 4 test lattice, launches and latency are everything
        dict(name="bin_4x4", kind="bin", l1=4, l2=4, beta=5.0),
        # the benchmark's headline chain
        dict(name="chain_16x16", kind="chain", l1=16, l2=16, beta=10.0),
        # the benchmark's complex hopping: two orbitals, Ndim 288, Ltrot 120, flux pi/4 per plaquette
        dict(name="chain_honeycomb_flux", kind="chain", lattice="Honeycomb", l1=12, l2=12, beta=12.0, u=3.0, nwrap=8,
             flux=18),
        # a large single chain of the serving stream, on the Hubbard plugin's default hopping
        dict(name="chain_24x24_checkerboard", kind="chain", l1=24, l2=24, beta=4.0, checkerboard=True),
        # production measurement: equal-time and time-displaced observables after each sweep
        dict(name="bin_16x16_tau", kind="bin", l1=16, l2=16, beta=10.0, tau=True),
        # the batched headline: 256 walkers of the benchmark's model on one device (the largest)
        dict(name="batch256_16x16", kind="batch", l1=16, l2=16, beta=10.0, chains=256),
        # a batch on the checkerboard hopping
        dict(name="batch64_16x16_checkerboard", kind="batch", l1=16, l2=16, beta=10.0, chains=64, checkerboard=True),
        # the mixed-precision form of the hopping wraps
        dict(name="batch64_16x16_split", kind="batch", l1=16, l2=16, beta=10.0, chains=64, split=True),
        # many small walkers, a few sweeps between reads
        dict(name="batch256_4x4", kind="batch", l1=4, l2=4, beta=5.0, chains=256, sweeps=10),
        # a temperature scan on an odd-sized lattice (Ndim 99): one batch of uneven Ltrot
        dict(name="batch32_9x11_uneven", kind="batch", l1=9, l2=11, beta=10.0, beta_min=2.0, chains=32),
        # a host that drives the slices itself
        dict(name="segment_16x16", kind="segment", l1=16, l2=16, beta=10.0),
        # the largest lattice: start from a new configuration (a restart, an admitted request)
        dict(name="init_32x32_checkerboard", kind="init", l1=32, l2=32, beta=4.0, checkerboard=True),
    ]
    return [{**base, **r} for r in rows]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges (no name), no dearer than the largest listed one."""
    kind = rng.choice(["chain", "chain", "bin", "batch", "batch", "segment", "init"])
    c = {"lattice": "Square", "nwrap": 10, "flux": 0, "checkerboard": False, "chains": 1, "split": False,
         "tau": False, "beta_min": 0.0, "sweeps": 1, "kind": kind, "u": round(rng.uniform(2.0, 8.0), 2)}
    top = {"chain": 20, "bin": 14, "batch": 16, "segment": 20, "init": 26}[kind]
    c["l1"] = _log_int(rng, 4, top)
    c["l2"] = min(top, max(4, c["l1"] + rng.choice([-2, -1, 0, 0, 1, 2])))
    c["beta"] = round(rng.uniform(2.0, 12.0 if c["l1"] * c["l2"] <= 320 else 5.0), 1)
    if rng.random() < 0.25 and c["l1"] <= 12 and kind != "bin":
        c.update(lattice="Honeycomb", nwrap=8, flux=rng.choice([0, 1, 3]), l2=c["l1"])
    if rng.random() < 0.35:
        c["checkerboard"] = True
        if c["lattice"] == "Square":            # the square families need even lengths
            c["l1"] += c["l1"] % 2
            c["l2"] += c["l2"] % 2
    if kind == "bin":
        c["tau"] = rng.random() < 0.4
    if kind == "batch":
        # at most a quarter of the largest listed batch's n^3 L chains, and little to set up
        n = c["l1"] * c["l2"] * (2 if c["lattice"] == "Honeycomb" else 1)
        room = 0.25 * 256 * 256 ** 3 * 10.0 / (n ** 3 * c["beta"])
        c["chains"] = max(2, min(_log_int(rng, 3, 160), int(room)))
        if not c["checkerboard"]:
            pick = rng.random()
            if pick < 0.3:
                c["beta_min"] = 2.0 if c["beta"] > 2.5 else 0.0
            elif pick < 0.5:
                c["split"] = True
    return c


@lru_cache(maxsize=None)
def _model(lattice, l1, l2, beta, u, nwrap, flux, checkerboard):
    """The host model (its set-up depends on the parameters alone)."""
    return hubbard_ham_set(HubbardParams(Lattice_type=lattice, L1=l1, L2=l2, Beta=beta, Dtau=0.1, Ham_U=u,
                                         Nwrap=nwrap, N_Phi=flux, Checkerboard=checkerboard))


def _betas(case):
    """Inverse temperature of each chain: one value, or a scan of whole slices."""
    b = case["chains"]
    if not case["beta_min"]:
        return [case["beta"]] * b
    return [round(x, 1) for x in np.linspace(case["beta_min"], case["beta"], b)]


def _models(case):
    return [_model(case["lattice"], case["l1"], case["l2"], beta, case["u"], case["nwrap"], case["flux"],
                   case["checkerboard"]) for beta in _betas(case)]


def _fields(n_op, ltrot, seed, chain=0):
    rng = np.random.default_rng([int(seed), chain])
    return FIELD_VALUES[rng.integers(0, 4, size=(n_op, ltrot))]


def _key(seed):
    return (int(seed) * 7919 + 17) % (1 << 48)


def prepare(case, seed):
    """A context with its fields and random stream, swept until its sweeps are replayed graphs
    (``chain``, ``bin``, ``batch``), with G at tau = 0 (``segment``), or as created (``init``)."""
    models = _models(case)
    kind = case["kind"]
    if kind == "batch":
        eng = BatchEngine(models)
        if case["split"]:
            eng.set_precision(PREC_INT8_SPLIT)
        for z, m in enumerate(models):
            eng.chain(z).set_fields(_fields(m.n_op, m.Ltrot, seed, z))
            eng.set_philox(_key(seed), z)
    else:
        eng = Engine(models[0])
        eng.set_fields(_fields(models[0].n_op, models[0].Ltrot, seed))
        eng.set_philox(_key(seed), 0)
    state = {"case": case, "eng": eng, "models": models}
    if kind == "init":
        state["fields"] = _fields(models[0].n_op, models[0].Ltrot, seed)
        return state
    if kind == "bin":
        eng.obs_setup()
    eng.init()
    if kind == "segment":
        return state
    if kind == "bin":
        eng.obs_enable(True)
        if case["tau"]:
            eng.tau_enable(True)
    eng.sweep(WARM[kind])
    if kind == "bin":
        eng.obs_reset()
    return state


def run(state):
    """One pass; the engine's state advances as in a running simulation."""
    case, eng = state["case"], state["eng"]
    kind = case["kind"]
    if kind == "init":
        eng.set_fields(state["fields"])
        eng.init()
        return {"green": eng.get_green(), "phase": _pair(eng.get_phase())}
    if kind == "segment":
        w = min(case["nwrap"], state["models"][0].Ltrot)
        phases = []
        for nt in range(w):
            phases.append(eng.wrapgrup(nt, eng.get_phase()))
        eng.wrapur(0, w)
        eng.udv_assign(ALFQ_UDVL, 1)
        eng.cgr(1, check_precision=True)
        for nt in range(w, 0, -1):
            phases.append(eng.wrapgrdo(nt, eng.get_phase()))
        eng.wrapul(w, 0)
        eng.udv_reset(ALFQ_UDVR, "R")
        eng.cgr(1, check_precision=True)
        return {"green": eng.get_green(), "phases": np.array(phases), "fields": eng.get_fields(),
                "position": eng.rng_position()}
    eng.sweep(case["sweeps"])
    if kind == "batch":
        out = []
        for z in range(case["chains"]):
            eng.chain(z)
            out.append((eng.get_green(), eng.get_phase(), eng.get_fields()))
        eng.chain(0)
        return {"green": np.stack([o[0] for o in out]), "phase": np.array([o[1] for o in out]),
                "fields": np.concatenate([o[2].ravel() for o in out])}
    got = {"green": eng.get_green(), "phase": _pair(eng.get_phase()), "fields": eng.get_fields()}
    if kind == "bin":
        s = eng.obs_get()
        got["obs"] = {k: s[k] for k in ("scal", "latt", "den0", "sign_scal", "n_scal")}
        if case["tau"]:
            t = eng.tau_get()
            got["tau"] = {k: t[k] for k in ("latt", "den0", "n")}
    return got


def _pair(z):
    return np.array([z.real, z.imag])


# ---- the work of a pass --------------------------------------------------------------------

ACCEPTANCE = 0.35


def work(case):
    """Algorithmic flops of the sweep (wraps 6 L c_T n^3, or 28 flops per bond and column on the
    checkerboard; UDV, QR and solves 117.3 S n^3; rank-1 updates 16 acc L n^3) and its inputs and
    outputs, each once."""
    flops = byts = 0.0
    per_cell = 2 if case["lattice"] == "Honeycomb" else 1
    n = case["l1"] * case["l2"] * per_cell
    hop = (28.0 * (3 if per_cell == 2 else 2) / per_cell * n ** 2 if case["checkerboard"]
           else (8.0 if case["flux"] else 4.0) * n ** 3)
    for beta in _betas(case):
        sl = int(round(beta / 0.1))
        s = -(-sl // case["nwrap"])
        if case["kind"] == "init":
            flops += sl * hop + (s + 1) * 58.0 * n ** 3
        elif case["kind"] == "segment":
            w = min(case["nwrap"], sl)
            flops += 6 * w * hop + 117.3 * n ** 3 + 16 * ACCEPTANCE * w * n ** 3
        else:
            f = 6 * sl * hop + 117.3 * s * n ** 3 + 16 * ACCEPTANCE * sl * n ** 3
            if case["tau"]:
                f += 4 * sl * hop + s * 8 * 8 * n ** 3 * 8.0 / 3.0
            flops += f * case["sweeps"]
        byts += 2 * 16.0 * n ** 2 + 2.0 * n * sl + (0 if case["checkerboard"] else 16.0 * n ** 2)
        if case["tau"]:
            byts += 3 * 16.0 * (sl + 1) * n
    return {"bytes": byts, "flops": flops}


# ---- the same quantities from plain numpy, for the sizes where that is quick -----------------

def _hop_square(l1, l2):
    """Nearest-neighbour hopping (t = 1) of the periodic lattice, cells in row-major order."""
    o = np.zeros((l1 * l2, l1 * l2))
    site = lambda i, j: (i % l1) * l2 + j % l2  # noqa: E731
    for i in range(l1):
        for j in range(l2):
            for k in (site(i + 1, j), site(i, j + 1)):
                o[site(i, j), k] = o[k, site(i, j)] = -1.0
    return o


def _exp_hop(case, sign):
    """exp(-sign dtau T): dense, or the ordered product of the four checkerboard families."""
    l1, l2, g = case["l1"], case["l2"], -sign * 0.1
    n = l1 * l2
    if not case["checkerboard"]:
        e, v = np.linalg.eigh(_hop_square(l1, l2))
        return (v * np.exp(g * e)) @ v.T
    ch, sh = math.cosh(0.1), math.sinh(0.1) * sign
    order = []
    for parity in (0, 1):
        for d in ((0, 1), (1, 0)):
            fam = []
            for i in range(l1):
                for j in range(l2):
                    if (i + j - (l1 - 1) // 2 - (l2 - 1) // 2) % 2 == parity:
                        fam.append((i * l2 + j, (i + d[0]) % l1 * l2 + (j + d[1]) % l2))
            order.append(np.array(fam))
    m = np.eye(n)
    for fam in (reversed(order) if sign > 0 else order):
        a, b = m[fam[:, 0]], m[fam[:, 1]]
        m[fam[:, 0]], m[fam[:, 1]] = ch * a + sh * b, ch * b + sh * a
    return m


_S6 = math.sqrt(6.0)
_PHI = {-2: -math.sqrt(2 * (3 + _S6)), -1: -math.sqrt(2 * (3 - _S6)), 1: math.sqrt(2 * (3 - _S6)),
        2: math.sqrt(2 * (3 + _S6))}
_GAMA = {-2: 1 - _S6 / 3, -1: 1 + _S6 / 3, 1: 1 + _S6 / 3, 2: 1 - _S6 / 3}
_FLIP = {-2: (-1, 1, 2), -1: (1, 2, -2), 1: (2, -2, -1), 2: (-2, -1, 1)}


class _Walk:
    """One chain of the square-lattice model in numpy: exp(V) exp(-dtau T) per slice."""

    def __init__(self, case, seed):
        self.n = case["l1"] * case["l2"]
        self.sl = int(round(case["beta"] / 0.1))
        self.w = case["nwrap"]
        self.et, self.eti = _exp_hop(case, 1), _exp_hop(case, -1)
        self.g = 1j * math.sqrt(0.1 * case["u"] / 2)
        self.f = _fields(self.n, self.sl, seed).copy()
        self.key, self.pos, self.phase = _key(seed), 0, 1.0 + 0j
        self.phi = np.array([_PHI.get(k, 0.0) for k in range(-2, 3)])

    def d(self, nt):
        return np.exp(self.g * self.phi[self.f[:, nt] + 2])

    def _left(self, hi, lo, state):
        """(U, D, V) of B(hi) ... B(lo + 1), one graded QR per interval, smallest slice last."""
        u, dd, v = state
        for nt in range(lo, hi):
            u = self.d(nt)[:, None] * (self.et @ u)
        a = u * dd
        p = np.argsort(-np.linalg.norm(a, axis=0), kind="stable")
        q, r = np.linalg.qr(a[:, p])
        dd = np.abs(np.diag(r))
        return q, dd, (r / dd[:, None]) @ v[p]

    def green(self, at):
        """(1 + B(at) ... B(1) B(L) ... B(at + 1))^-1 and the phase of its weight."""
        one = np.eye(self.n, dtype=complex)
        state = (one, np.ones(self.n), one)
        for lo, hi in ((at, self.sl), (0, at)):
            for k in range(lo, hi, self.w):
                state = self._left(min(k + self.w, hi), k, state)
        u, dd, v = state
        big, small = np.where(dd > 1, 1 / dd, 1.0), np.where(dd > 1, 1.0, dd)
        m = big[:, None] * u.conj().T + small[:, None] * v
        z = np.linalg.slogdet(m)[0] * np.linalg.slogdet(u)[0]
        z *= np.exp(1j * (self.g * -0.5).imag * self.phi[self.f + 2].sum())
        return np.linalg.solve(m, big[:, None] * u.conj().T), z * z

    def uniforms(self, count):
        """The next `count` numbers of the Philox4x32-10 stream (one block each, 53 bits)."""
        q = np.arange(self.pos, self.pos + count, dtype=np.uint64)
        self.pos += count
        low = np.uint64(0xFFFFFFFF)
        c = [q & low, q >> np.uint64(32), np.zeros_like(q), np.full_like(q, 0x414C4651)]
        k0, k1 = self.key & 0xFFFFFFFF, self.key >> 32
        for _ in range(10):
            a, b = c[0] * np.uint64(0xD2511F53), c[2] * np.uint64(0xCD9E8D57)
            c = [(b >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), b & low, (a >> np.uint64(32)) ^ c[3] ^ np.uint64(k1),
                 a & low]
            k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
        return (((c[0] << np.uint64(32)) | c[1]) >> np.uint64(11)).astype(np.float64) / 2.0 ** 53

    def metropolis(self, g, nt, order):
        u = self.uniforms(3 * self.n)
        for k, p in enumerate(order):
            old = int(self.f[p, nt])
            new = _FLIP[old][min(max(int(math.floor(3 * u[3 * k] + 1.0)), 1), 3) - 1]
            z1 = self.g * (_PHI[new] - _PHI[old])
            e = np.exp(z1)
            ratio = ((e - (e - 1) * g[p, p]) * np.exp(-0.5 * z1)) ** 2 * _GAMA[new] / _GAMA[old]
            if abs((self.phase * ratio).real / self.phase.real) <= u[3 * k + 2]:
                continue
            self.phase *= ratio / abs(ratio)
            v = -g[p]
            v[p] += 1
            g -= np.outer(g[:, p], (e - 1) / (1 + v[p] * (e - 1)) * v)
            self.f[p, nt] = new

    def up(self, g, nt):
        g = self.et @ g @ self.eti
        d = self.d(nt)
        g = d[:, None] * g / d
        self.metropolis(g, nt, range(self.n))
        return g

    def down(self, g, nt):
        self.metropolis(g, nt, range(self.n - 1, -1, -1))
        d = self.d(nt)
        return self.eti @ (g / d[:, None] * d) @ self.et

    def sweep(self, g, seen=None):
        stops = set(range(0, self.sl, self.w)) | {self.sl}
        for nt in range(self.sl):
            g = self.up(g, nt)
            if nt + 1 in stops:
                g, self.phase = self.green(nt + 1)
            if seen is not None:
                seen(g, self.phase)
        for nt in range(self.sl - 1, -1, -1):
            g = self.down(g, nt)
            if seen is not None and nt > 0:      # measured on slices 1 .. Ltrot
                seen(g, self.phase)
            if nt in stops:
                g, self.phase = self.green(nt)
        return g


def exact(case, seed):
    """The floating outputs of `run` on a new state from numpy, or None where that is slow (long
    or large chains, batches) or the model is not the plain square lattice."""
    kind, n = case["kind"], case["l1"] * case["l2"]
    if case["lattice"] != "Square" or case["flux"] or kind == "batch" or case["tau"] or min(case["l1"], case["l2"]) < 3:
        return None
    if kind in ("chain", "bin") and (n > 36 or (case["checkerboard"] and kind == "bin")):
        return None
    if n * n * n * case["beta"] > 5e9:
        return None
    wk = _Walk(case, seed)
    g, wk.phase = wk.green(0)
    if kind == "init":
        return {"green": g, "phase": _pair(wk.phase)}
    if kind == "segment":
        w, phases = min(wk.w, wk.sl), []
        for nt in range(w):
            g = wk.up(g, nt)
            phases.append(wk.phase)
        g, wk.phase = wk.green(w)
        for nt in range(w - 1, -1, -1):
            g = wk.down(g, nt)
            phases.append(wk.phase)
        g, _ = wk.green(0)
        return {"green": g, "phases": np.array(phases), "fields": None, "position": None}
    for _ in range(WARM[kind]):
        g = wk.sweep(g)
    scal = np.zeros(4, dtype=complex)
    hop = _hop_square(case["l1"], case["l2"])

    def seen(gr, phase):
        zs = np.sign(phase.real)
        grc = np.eye(n) - gr.T
        kin, dens = 2 * np.sum(hop * grc), np.diag(grc)
        pot = case["u"] * np.sum(dens * dens)
        scal[:] += np.array([kin, pot, 2 * dens.sum(), kin + pot]) * zs * phase / phase.real

    for _ in range(case["sweeps"]):
        g = wk.sweep(g, seen)
    got = {"green": g, "phase": _pair(wk.phase), "fields": None}
    if kind == "bin":
        got["obs"] = {"scal": scal, "latt": None, "den0": None, "sign_scal": None, "n_scal": None}
    return got
