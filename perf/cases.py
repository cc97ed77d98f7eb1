"""The workloads that timing runs of this framework use, through its Python
front end (vegas-rs_amd/__init__.py): batches of lattice chains, Wolff chains,
chains over an exchange matrix, and the job server.

listed() names them, draw() gives more of the same ranges, prepare() makes
what a program holds before the call (its batch or server, spins from the
chain seeds, thermostats), run() is one pass and returns what the call
returns, work() what a pass cannot do without, and exact() the observables of
the Metropolis Ising passes, from numpy in 64 bits.
"""
import importlib.util
import math
import sys
from pathlib import Path

import numpy as np

ROOT = Path(__file__).resolve().parents[1]

# Critical temperatures (J = 1) the temperature scans are centred on.
T_CRIT = {("sc", "ising"): 4.5115, ("bcc", "ising"): 6.3544, ("fcc", "ising"): 9.7937,
          ("sc", "heisenberg"): 1.443, ("bcc", "heisenberg"): 2.0542,
          ("fcc", "heisenberg"): 3.1757}
SITES_PER_CELL = {"sc": 1, "bcc": 2, "fcc": 4}
MIXED_SIDES = (16, 24, 32, 48, 64, 96, 128)  # the mixed-size batch of bench.py
RELAX = 4        # sweeps run while preparing, so that a pass does not start from infinite T
EXACT_LIMIT = 12_000_000  # attempts that exact() is willing to repeat in numpy


def _sim(name, lattice, spin, proposal, dims, sweeps, **more):
    case = {"name": name, "what": "chains", "lattice": lattice, "spin": spin,
            "proposal": proposal, "lx": dims[0], "ly": dims[1], "lz": dims[2], "open": "",
            "chains": 1, "mixed": 0, "sweeps": sweeps, "tuned": False, "snapshot": False,
            "field": 0.0, "anisotropy": 0.0, "compound": True}
    case.update(more)
    return case


def listed():
    return [
        # The command line's default input: 10x10x1, one chain; a stage of a
        # CoolDown is thousands of sweeps of a lattice that fits one wave.
        _sim("cli_10x10", "sc", "ising", "flip", (10, 10, 1), 1000, open="z"),
        # The smallest call: a Machine stepped one sweep at a time (a hook or
        # a state snapshot after every step), odd sizes, one open axis.
        _sim("one_sweep_bcc", "bcc", "ising", "flip", (6, 5, 7), 1, open="z", field=0.1,
             snapshot=True),
        # `vegas bench heisenberg 16`: bare Exchange, fresh proposals, and the
        # state written out at the end of the stage.
        _sim("bench_heis_16", "sc", "heisenberg", "random", (16, 16, 16), 200, compound=False,
             snapshot=True),
        # A temperature and field scan of uneven sizes in one batch, replayed
        # from captured sweep blocks: the mixed-size set of bench.py, a
        # quarter of it.
        _sim("scan_mixed_128", "sc", "ising", "flip", (0, 0, 0), 50, chains=128, mixed=2024,
             field=0.1, tuned=True),
        # Jobs served together: short Relax, CoolDown and HysteresisLoop jobs
        # of the served mix's sizes.
        {"name": "served_24", "what": "served", "jobs": 24, "mixed": 2025, "sweeps": 100,
         "stage_sweeps": 20},
        # The headline: three chains of 256^3, int8, tuned and replayed.
        _sim("sc_256x3", "sc", "ising", "flip", (256, 256, 256), 100, chains=3, tuned=True,
             compound=False),
        # The largest lattice, one bit per site, fresh proposals.
        _sim("sc_1024_bits", "sc", "bits", "random", (1024, 1024, 1024), 4),
        # bcc ensemble at the size bench.py measures.
        _sim("bcc_160x3", "bcc", "ising", "flip", (160, 160, 160), 50, chains=3, tuned=True,
             compound=False),
        # A film: fcc, ragged sizes, open along z, plain launches, and the
        # state written out after the block (StateSensor).
        _sim("fcc_film", "fcc", "ising", "flip", (125, 90, 61), 50, open="z", field=0.05,
             snapshot=True),
        # Heisenberg at its bench size: anisotropy and field, fresh proposals.
        _sim("heis_128x3", "sc", "heisenberg", "random", (128, 128, 128), 20, chains=3,
             field=0.05, anisotropy=0.1, tuned=True),
        # Wolff cluster steps at T_c, many chains.
        _sim("wolff_32x64", "sc", "ising", "wolff", (32, 32, 32), 40, chains=64,
             compound=False),
        # A spin glass: +-J couplings given as a sparse matrix, with its state.
        {"name": "glass_32", "what": "matrix", "spin": "ising", "proposal": "flip", "side": 32,
         "sweeps": 100, "snapshot": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["small", "small", "step", "single", "scan", "ensemble", "film", "heis",
                       "heis", "wolff", "matrix", "served", "large"])
    lattice = rng.choice(["sc", "bcc", "fcc"])
    proposal = rng.choice(["flip", "random"])
    opened = rng.choice(["", "", "z", "xy"])

    def dims(lo, hi):
        d = [max(2, _log_int(rng, lo, hi)) for _ in range(3)]
        if lattice == "sc":  # an even x length, even periodic axes
            d = [v + v % 2 for v in d]
        return d

    if kind == "small":  # one chain of the sizes a person runs by hand
        spin = rng.choice(["ising", "heisenberg"])
        return _unnamed(_sim("", lattice, spin, proposal, dims(4, 24), _log_int(rng, 50, 1000),
                             open=opened, field=rng.choice([0.0, 0.1])))
    if kind == "step":
        spin = rng.choice(["ising", "bits", "heisenberg"])
        return _unnamed(_sim("", lattice, spin, proposal, dims(4, 40), rng.randint(1, 4),
                             open=opened, snapshot=rng.random() < 0.5))
    if kind == "single":  # one chain, between the hand-run and the largest sizes
        spin = rng.choice(["ising", "bits"])
        return _unnamed(_sim("", lattice, spin, proposal, dims(24, 160), _log_int(rng, 10, 200),
                             open=opened, tuned=rng.random() < 0.5))
    if kind == "scan":
        return _unnamed(_sim("", "sc", rng.choice(["ising", "bits"]), proposal, (0, 0, 0),
                             rng.randint(10, 50), chains=rng.randint(8, 128),
                             mixed=rng.randint(1, 9999), field=0.1, tuned=rng.random() < 0.5))
    if kind == "ensemble":
        spin = rng.choice(["ising", "ising", "bits"])
        d = dims(64, 256) if lattice == "sc" else dims(40, 128)
        return _unnamed(_sim("", lattice, spin, proposal, d, rng.randint(10, 50),
                             chains=rng.randint(2, 4), tuned=True, compound=False))
    if kind == "film":
        d = dims(24, 120)
        d[2] = max(2, d[2] // 2 + (d[2] // 2) % 2)
        return _unnamed(_sim("", lattice, rng.choice(["ising", "bits"]), "flip", d,
                             rng.randint(10, 60), open="z", field=0.05, snapshot=True))
    if kind == "heis":
        return _unnamed(_sim("", lattice, "heisenberg", proposal,
                             dims(12, 128) if lattice == "sc" else dims(12, 70),
                             rng.randint(4, 40), chains=rng.randint(1, 3), open=opened,
                             field=rng.choice([0.0, 0.05]), anisotropy=rng.choice([0.0, 0.1]),
                             tuned=rng.random() < 0.5))
    if kind == "wolff":
        d = dims(8, 40) if lattice == "sc" else dims(6, 20)
        return _unnamed(_sim("", lattice, "ising", "wolff", d, rng.randint(5, 40),
                             chains=rng.randint(1, 64), compound=False))
    if kind == "matrix":
        return {"what": "matrix", "spin": rng.choice(["ising", "heisenberg"]),
                "proposal": proposal, "side": 2 * rng.randint(4, 24),
                "sweeps": rng.randint(10, 100), "snapshot": rng.random() < 0.5}
    if kind == "served":
        return {"what": "served", "jobs": rng.randint(4, 24), "mixed": rng.randint(1, 9999),
                "sweeps": rng.randint(20, 100), "stage_sweeps": rng.randint(5, 20)}
    side = 2 * _log_int(rng, 128, 400)
    return _unnamed(_sim("", "sc", rng.choice(["ising", "bits"]), proposal, (side, side, side),
                         rng.randint(1, 4)))


def _unnamed(case):
    del case["name"]
    return case


# ---------------------------------------------------------------- the calls

def _engine():
    if "vegas_hip" not in sys.modules:
        spec = importlib.util.spec_from_file_location("vegas_hip",
                                                      ROOT / "vegas-rs_amd" / "__init__.py")
        mod = importlib.util.module_from_spec(spec)
        sys.modules["vegas_hip"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["vegas_hip"]


_contexts = []


def _context():
    if not _contexts:
        _contexts.append(_engine().Context(0))
    return _contexts[0]


class Held:
    """A batch or server that is closed with its last reference."""

    def __init__(self, handle, **more):
        self.handle = handle
        self.__dict__.update(more)

    def __del__(self):
        self.handle.close()


def _chains_of(case):
    """(dims, temperature, field, field direction) of every chain of a case."""
    tc = T_CRIT[case["lattice"], "heisenberg" if case["spin"] == "heisenberg" else "ising"]
    n = case["chains"]
    if case["mixed"]:
        pick = np.random.default_rng(case["mixed"])
        sides = pick.choice(np.array(MIXED_SIDES), size=n)
        temps = pick.uniform(3.5, 5.5, size=n)
        fields = pick.uniform(-case["field"], case["field"], size=n)
        return [((int(s),) * 3, float(t), abs(float(h)), 1.0 if h >= 0 else -1.0)
                for s, t, h in zip(sides, temps, fields)]
    dims = (case["lx"], case["ly"], case["lz"])
    if case["proposal"] == "wolff" or n == 1:
        temps = [tc] * n
    else:
        temps = [float(t) for t in np.linspace(0.78 * tc, 1.33 * tc, n)]
    return [(dims, t, case["field"], 1.0) for t in temps]


def _chain_seed(seed, k):
    return (int(seed) * 1000003 + k) & 0xFFFFFFFFFFFF


def prepare(case, seed):
    vg, ctx = _engine(), _context()
    if case["what"] == "served":
        jobs = _served_jobs(vg, case, seed)
        return Held(vg.Server(ctx, memory_bytes=1 << 28, max_jobs=64, quantum_sweeps=50),
                    case=case, jobs=jobs)
    if case["what"] == "matrix":
        matrix = _glass(case["side"], seed)
        spin = vg.ISING if case["spin"] == "ising" else vg.HEISENBERG
        prop = vg.FLIP if case["proposal"] == "flip" else vg.RANDOM
        desc = vg.chain(vg.graph_lattice(), spin, prop,
                        vg.hamiltonian(exchange=1.0, zeeman=True), _chain_seed(seed, 0))
        b = vg.Batch(ctx, [desc], exchange=[matrix])
        b.randomize()
        b.set_thermostat(0, 1.1)
        b.run(RELAX, observe=False)
        return Held(b, case=case)
    kind = {"sc": vg.SC, "bcc": vg.BCC, "fcc": vg.FCC}[case["lattice"]]
    spin = {"ising": vg.ISING, "bits": vg.ISING_BITS, "heisenberg": vg.HEISENBERG}[case["spin"]]
    prop = {"flip": vg.FLIP, "random": vg.RANDOM, "wolff": vg.WOLFF}[case["proposal"]]
    pbc = tuple(axis not in case["open"] for axis in "xyz")
    more = {"anisotropy": case["anisotropy"]} if case["anisotropy"] else {}
    ham = vg.hamiltonian(exchange=1.0, zeeman=case["compound"], **more)
    chains = _chains_of(case)
    descs = [vg.chain(vg.lattice(kind, *dims, pbc=pbc), spin, prop, ham, _chain_seed(seed, k))
             for k, (dims, _, _, _) in enumerate(chains)]
    b = vg.Batch(ctx, descs)
    b.randomize()
    for k, (dims, t, field, up) in enumerate(chains):
        b.set_thermostat(k, t, field, (0.0, 0.0, up))
        if case["proposal"] == "wolff":  # from the ordered state: clusters of T_c's sizes
            n = SITES_PER_CELL[case["lattice"]] * dims[0] * dims[1] * dims[2]
            b.set_ising(k, np.ones(n, dtype=np.int8))
    if case["tuned"]:
        b.autotune(6)
        b.set_graph(True)
        b.prepare(case["sweeps"])
    b.run(40 if case["proposal"] == "wolff" else RELAX, observe=False)
    return Held(b, case=case)


def _served_jobs(vg, case, seed):
    """60% Ising Relax, 30% Heisenberg CoolDown, 10% Heisenberg HysteresisLoop
    (bench.py's served mix with fewer sweeps and stages)."""
    pick = np.random.default_rng(case["mixed"])
    ising = vg.hamiltonian(exchange=1.0, zeeman=True)
    heis = vg.hamiltonian(exchange=1.0, zeeman=True, anisotropy=0.1)
    jobs = []
    for k in range(case["jobs"]):
        u, side, t = pick.random(), int(pick.integers(8, 49)) * 2, float(pick.uniform(2.0, 6.0))
        hside = int(pick.integers(8, 25)) * 2
        s = _chain_seed(seed, k)
        if u < 0.6:
            jobs.append((vg.chain(vg.lattice(vg.SC, side, side, side), vg.ISING, vg.FLIP, ising,
                                  s), vg.relax(case["sweeps"], t)))
        elif u < 0.9:
            jobs.append((vg.chain(vg.lattice(vg.SC, hside, hside, hside), vg.HEISENBERG,
                                  vg.RANDOM, heis, s),
                         vg.cool_down(3.0, 0.6, 0.6, relax=0, steps=case["stage_sweeps"])))
        else:
            jobs.append((vg.chain(vg.lattice(vg.SC, 32, 32, 32), vg.HEISENBERG, vg.RANDOM, heis,
                                  s),
                         vg.hysteresis_loop(steps=case["stage_sweeps"], relax=0, temperature=1.0,
                                            max_field=0.5, field_step=0.5)))
    return jobs


def _glass(side, seed):
    """Edwards-Anderson couplings: +-1 on the bonds of a periodic side^3
    cubic lattice, as CSR (row_ptr, col, value)."""
    rng = np.random.default_rng([int(seed), side])
    n = side ** 3
    ids = np.arange(n).reshape(side, side, side)
    col, val = np.empty((n, 6), dtype=np.uint64), np.empty((n, 6))
    for axis in range(3):
        j = rng.choice(np.array([-1.0, 1.0]), size=(side, side, side))
        col[:, 2 * axis] = np.roll(ids, -1, axis).reshape(n)
        val[:, 2 * axis] = j.reshape(n)
        col[:, 2 * axis + 1] = np.roll(ids, 1, axis).reshape(n)
        val[:, 2 * axis + 1] = np.roll(j, 1, axis).reshape(n)
    return np.arange(n + 1, dtype=np.uint64) * np.uint64(6), col.reshape(-1), val.reshape(-1)


def run(state):
    case, h = state.case, state.handle
    if case["what"] == "served":
        ids = [h.submit(d, stages) for d, stages in state.jobs]
        lines, last = [], []
        for jid in ids:
            st = h.wait(jid)
            last.append((st.last_energy, st.last_magnetization))
            lines.append(h.results(jid))
            h.release(jid)
        return {"stages": np.concatenate(lines), "last": np.array(last)}
    e, m = h.run(case["sweeps"])
    out = {"energy": e, "magnetization": m}
    if case.get("snapshot"):
        get = h.get_heisenberg if case["spin"] == "heisenberg" else h.get_ising
        out["spins"] = [get(i) for i in range(h.n)]
    return out


def _attempts(case):
    """Single-site attempts of one pass (Wolff: none)."""
    if case["what"] == "matrix":
        return case["side"] ** 3 * case["sweeps"]
    sites = sum(SITES_PER_CELL[case["lattice"]] * d[0] * d[1] * d[2]
                for d, _, _, _ in _chains_of(case))
    return sites * case["sweeps"]


# Bytes of one attempt: the site's spin read and written.
SITE_BYTES = {"ising": 2.0, "bits": 0.25, "heisenberg": 24.0}


def work(case):
    """Every spin read and written once per sweep, the observables written;
    arithmetic of the neighbour sums, the energy difference and the
    acceptance.  Wolff: the flipped sites at T_c (bench.py's mean cluster)."""
    if case["what"] == "served":
        vg = _engine()
        by = fl = 0.0
        for d, stages in _served_jobs(vg, case, 0):
            n = d.lattice.lx * d.lattice.ly * d.lattice.lz * sum(s.relax + s.measure
                                                                 for s in stages)
            heis = d.spin == vg.HEISENBERG
            by += n * SITE_BYTES["heisenberg" if heis else "ising"]
            fl += n * (90 if heis else 12)
        return {"bytes": by, "flops": fl}
    if case["what"] == "matrix":
        per = 6 * 12 + SITE_BYTES[case["spin"]]  # a row's columns and couplings, the spin
        n = _attempts(case)
        return {"bytes": n * per, "flops": n * (90 if case["spin"] == "heisenberg" else 30)}
    z = {"sc": 6, "bcc": 8, "fcc": 12}[case["lattice"]]
    observed = 16.0 * case["chains"] * case["sweeps"]
    if case["proposal"] == "wolff":
        n = SITES_PER_CELL[case["lattice"]] * case["lx"] * case["ly"] * case["lz"]
        flipped = 916.0 * (n / 32768.0) ** 0.654 * case["chains"] * case["sweeps"]
        return {"bytes": flipped * (2 + z) + observed, "flops": flipped * z * 4}
    n = _attempts(case)
    flops = 3 * z + 70 if case["spin"] == "heisenberg" else z + 6
    out = 0.0
    if case["snapshot"]:
        out = n / case["sweeps"] * (24.0 if case["spin"] == "heisenberg" else 1.0)
    return {"bytes": n * SITE_BYTES[case["spin"]] + observed + out, "flops": float(n * flops)}


# -------------------------------------------- the same observables in numpy

def _philox(x, y, z, w, seed):
    """Philox4x32-10 (Salmon et al., SC'11) of uint32 counter arrays."""
    m0, m1, low = np.uint64(0xD2511F53), np.uint64(0xCD9E8D57), np.uint64(0xFFFFFFFF)
    s32 = np.uint64(32)
    x, y, z, w = (np.asarray(v, dtype=np.uint64) for v in np.broadcast_arrays(x, y, z, w))
    k0, k1 = seed & 0xFFFFFFFF, seed >> 32
    for _ in range(10):
        p0, p1 = x * m0, z * m1
        x, y, z, w = (p1 >> s32) ^ y ^ np.uint64(k0), p1 & low, \
            (p0 >> s32) ^ w ^ np.uint64(k1), p0 & low
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return np.stack([x, y, z, w])


def _word(sweep, purpose, colour):
    return ((sweep >> 32) << 8) | ((colour >> 1) << 7) | (purpose << 1) | (colour & 1)


class _Checkerboard:
    """One Ising chain: colour planes of +-1 over [z][y][position]."""

    def __init__(self, case, dims, t, field, up, seed):
        self.kind, self.random, self.seed = case["lattice"], case["proposal"] == "random", seed
        self.lx, self.ly, self.lz = dims
        self.periodic = [a not in case["open"] for a in "xyz"]
        self.t, self.field, self.up, self.compound = t, field, up, case["compound"]
        self.colours = 4 if self.kind == "fcc" else 2
        self.w = self.lx // 2 if self.kind == "sc" else self.lx
        self.pos = np.arange(self.w)
        self.row = (np.arange(self.ly)[None, :, None]
                    + self.ly * np.arange(self.lz)[:, None, None])
        self.parity = (np.arange(self.ly)[None, :, None] + np.arange(self.lz)[:, None, None]) & 1
        self.half = {"sc": None, "bcc": [0, 7], "fcc": [0, 6, 5, 3]}[self.kind]
        self.z = {"sc": 6, "bcc": 8, "fcc": 12}[self.kind]
        self.sweeps = 0
        self.planes = []
        for c in range(self.colours):
            r = _philox(self.pos >> 2, self.row, 0, _word(0, 3, c), seed)
            v = np.take_along_axis(r, np.broadcast_to(self.pos & 3, r.shape[1:])[None], 0)[0]
            self.planes.append(np.where(v < 1 << 31, 1, -1).astype(np.int64))

    def _move(self, a, axis, d):
        """a's value one cell along the axis (d = -1, 0, +1), 0 past an open end."""
        if d == 0:
            return a
        np_axis = 2 - axis
        a = np.roll(a, -d, np_axis)
        if not self.periodic[axis]:
            end = [slice(None)] * 3
            end[np_axis] = -1 if d > 0 else 0
            a = a.copy()
            a[tuple(end)] = 0
        return a

    def _neighbours(self, c, only_lower=False):
        """(sum of the present neighbours' spins, how many are present)."""
        total, there = 0, 0
        for b in range(self.colours):
            if b == c or (only_lower and b > c):
                continue
            for a, out in ((self.planes[b], 0), (np.ones_like(self.planes[b]), 1)):
                if self.kind == "sc":
                    q = (c + self.parity) & 1  # x of position i is 2 i + q
                    s = (a + np.where(q == 0, self._move(a, 0, -1), self._move(a, 0, 1))
                         + sum(self._move(a, ax, d) for ax in (1, 2) for d in (-1, 1)))
                else:
                    s = a
                    for ax in range(3):
                        mine, other = self.half[c] >> ax & 1, self.half[b] >> ax & 1
                        if mine != other:
                            s = s + self._move(s, ax, 1 if mine else -1)
                if out:
                    there = there + s
                else:
                    total = total + s
        return total, there

    def _high_byte(self, c):
        t = self.sweeps
        if self.kind != "sc":
            r = _philox(self.pos >> 4, self.row, t, _word(t, 0, c), self.seed)
            sel = np.broadcast_to((self.pos & 15) >> 2, r.shape[1:])
            return np.take_along_axis(r, sel[None], 0)[0] >> (8 * (self.pos & 3)).astype(
                np.uint64) & np.uint64(255)
        out = 0
        for half in range(2):
            r = _philox(2 * (self.pos >> 5) + half, self.row, t, _word(t, 0, c), self.seed)
            for k in range(4):
                bit = r[k] >> (self.pos & 31).astype(np.uint64) & np.uint64(1)
                out = out | bit << np.uint64(4 * half + k)
        return out

    def sweep(self):
        bond, t = 0, self.sweeps
        for c in range(self.colours):
            s = self.planes[c]
            sigma, _ = self._neighbours(c)
            hm = abs(self.field) if self.compound else 0.0
            de = 2.0 * s * sigma - 2.0 * hm * self.up * s
            th = np.ceil(np.exp(-np.maximum(de, 0.0) / self.t) * 2.0 ** 32)
            always = (de <= 0.0) | (th >= 2.0 ** 32)
            th = np.where(always, 0, th).astype(np.uint64)
            hi = self._high_byte(c)
            accept = always | (hi < th >> np.uint64(24))
            tied = np.argwhere(~always & (hi == th >> np.uint64(24)))
            if len(tied):
                zz, yy, i = tied.T
                r = _philox(i >> 2, yy + self.ly * zz, t, _word(t, 1, c), self.seed)
                lo = r[i & 3, np.arange(len(i))] >> np.uint64(8)
                accept[zz, yy, i] = lo < (th[zz, yy, i] & np.uint64(0xFFFFFF))
            if self.random:
                r = _philox(self.pos >> 7, self.row, t, _word(t, 2, c), self.seed)
                sel = np.broadcast_to((self.pos >> 5) & 3, r.shape[1:])
                down = (np.take_along_axis(r, sel[None], 0)[0]
                        >> (self.pos & 31).astype(np.uint64) & np.uint64(1))
                accept &= np.where(down == 0, 1, -1) != s
            self.planes[c] = np.where(accept, -s, s)
            if c:
                low, _ = self._neighbours(c, only_lower=True)
                bond += int((self.planes[c] * low).sum())
        self.sweeps += 1
        mag = sum(int(p.sum()) for p in self.planes)
        if self.compound:
            energy = -2.0 * bond + abs(self.field) * mag * self.up
        else:
            energy = -1.0 * bond
        return energy, float(abs(mag))

    def spins(self):
        """Natural site order, int8."""
        if self.kind == "sc":
            out = np.empty((self.lz, self.ly, self.lx), dtype=np.int8)
            for c in range(2):
                for p in range(2):
                    zz, yy = np.nonzero(self.parity[:, :, 0] == p)
                    out[zz, yy, (c + p) & 1::2] = self.planes[c][zz, yy]
            return out.reshape(-1)
        return np.stack(self.planes, axis=-1).astype(np.int8).reshape(-1)


def _exact_glass(case, seed):
    """The +-J chain: sites of a colour class at once (even sides: the parity
    classes), energies in f64."""
    side, t = case["side"], 1.1
    n = side ** 3
    _, col, val = _glass(side, seed)
    col, val = col.reshape(n, 6).astype(np.int64), val.reshape(n, 6)
    key, site = _chain_seed(seed, 0), np.arange(n)
    s = np.where(_philox(site, 0, 0, _word(0, 9, 0), key)[0] < 1 << 31, 1.0, -1.0)
    zz, yy, xx = site // side ** 2, site // side % side, site % side
    classes = [np.nonzero((xx + yy + zz) % 2 == c)[0] for c in range(2)]
    e, m = [], []
    for sweep in range(RELAX + case["sweeps"]):
        r = _philox(site, 0, sweep, _word(sweep, 8, 0), key)
        u = r[0] * 2.0 ** -32
        move = np.where(r[1] < 1 << 31, 1.0, -1.0) != s if case["proposal"] == "random" else None
        for cls in classes:
            de = 2.0 * s[cls] * (val[cls] * s[col[cls]]).sum(axis=1)
            accept = (de <= 0.0) | (u[cls] < np.exp(-np.maximum(de, 0.0) / t))
            if move is not None:
                accept &= move[cls]
            s[cls] = np.where(accept, -s[cls], s[cls])
        e.append(-(s[:, None] * val * s[col]).sum())
        m.append(abs(s.sum()))
    out = {"energy": np.array([e[RELAX:]]), "magnetization": np.array([m[RELAX:]])}
    if case["snapshot"]:
        out["spins"] = [s.astype(np.int8)]
    return out


def exact(case, seed):
    """Observables of the Ising Metropolis passes, repeated in numpy with the
    same keyed draws.  None for Heisenberg chains and Wolff steps (their
    trajectories follow the fp32 and bond-by-bond arithmetic), for the served
    mix, and for more than EXACT_LIMIT attempts."""
    if case["what"] == "served" or case["proposal"] == "wolff" or case["spin"] == "heisenberg":
        return None
    if _attempts(case) > EXACT_LIMIT:
        return None
    if case["what"] == "matrix":
        return _exact_glass(case, seed)
    es, ms, spins = [], [], []
    for k, (dims, t, field, up) in enumerate(_chains_of(case)):
        sim = _Checkerboard(case, dims, t, field, up, _chain_seed(seed, k))
        for _ in range(RELAX):
            sim.sweep()
        got = [sim.sweep() for _ in range(case["sweeps"])]
        es.append([g[0] for g in got])
        ms.append([g[1] for g in got])
        spins.append(sim.spins())
    out = {"energy": np.array(es), "magnetization": np.array(ms)}
    if case["snapshot"]:
        out["spins"] = spins
    return out
