"""Small Heisenberg chains, whose sweep blocks run in one workgroup each with
draws made beforehand: bit-exact against the CPU oracle at the edges of the
sites a lane takes, with open ends, both proposals, chains of different sizes
in one batch, and more sweeps than the workspace of draws holds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KINDS = {"sc": 0, "bcc": 1, "fcc": 2}


def _chain(vg, orc, kind, dims, pbc, proposal, seed, field):
    L = vg.lattice([vg.SC, vg.BCC, vg.FCC][KINDS[kind]], *dims, pbc=tuple(bool(p) for p in pbc))
    d = vg.chain(L, vg.HEISENBERG, vg.RANDOM if proposal == "random" else vg.FLIP,
                 vg.hamiltonian(exchange=1.0, anisotropy=0.2, zeeman=True), seed)
    OL = orc.lattice(kind, *dims, pbc=pbc)
    OM = orc.model(spin="heisenberg", proposal=proposal, terms=("exchange", "anisotropy", "zeeman"),
                   anisotropy=0.2, temperature=1.3, field=field)
    return d, OL, OM


def _check(vg, orc, ctx, chains, sweeps):
    with vg.Batch(ctx, [c[0] for c in chains]) as b:
        b.randomize()
        states = [orc.heis_init(c[1], c[3]) for c in chains]
        for k, c in enumerate(chains):
            b.set_thermostat(k, 1.3, c[4])
        done = 0
        for n in sweeps:
            got = b.run_sums(n)
            for k, (_, OL, OM, seed, _) in enumerate(chains):
                assert np.array_equal(got[k], orc.heis_sweeps(OL, OM, seed, done, n, states[k])), (n, k)
                assert np.array_equal(b.get_heisenberg(k), states[k].astype(np.float64)), (n, k)
            done += n


@pytest.mark.parametrize("kind,dims,pbc", [
    ("sc", (2, 2, 2), (1, 1, 1)), ("sc", (16, 4, 2), (1, 1, 1)), ("sc", (26, 5, 1), (1, 0, 0)),
    ("sc", (64, 8, 4), (1, 1, 1)), ("bcc", (41, 5, 5), (0, 1, 0)),   # 1024 and 1025 a colour
    ("bcc", (16, 16, 8), (1, 1, 1)), ("sc", (66, 8, 8), (1, 1, 1)),  # 2048 and 2112
    ("sc", (128, 8, 8), (1, 1, 1)), ("bcc", (17, 15, 16), (0, 0, 1)),  # 4096 and 4080: the largest
    ("fcc", (1, 1, 1), (1, 1, 1)), ("fcc", (9, 5, 23), (1, 0, 1)),   # 1 and 1035
    ("fcc", (16, 16, 8), (1, 1, 0)),                                 # 2048, the largest of fcc
])
def test_heis_resident_bit_exact(vg, orc, ctx, kind, dims, pbc):
    for proposal, field in (("random", 0.1), ("flip", -0.3)):
        d, OL, OM = _chain(vg, orc, kind, dims, pbc, proposal, 31, field)
        _check(vg, orc, ctx, [(d, OL, OM, 31, field)], (1, 7))


@pytest.mark.parametrize("kind,dims", [
    ("sc", [(32, 16, 16), (4, 4, 4), (10, 6, 8)]),
    ("fcc", [(12, 12, 13), (2, 3, 1)]),
])
def test_heis_resident_batches(vg, orc, ctx, kind, dims):
    """Eight chains of up to 8192 sites: the workspace holds 64 sweeps."""
    chains = []
    for k in range(8):
        prop = "flip" if k == 5 else "random"
        d, OL, OM = _chain(vg, orc, kind, dims[k % len(dims)], (1, 1, 1), prop, 90 + k, 0.05 * k)
        chains.append((d, OL, OM, 90 + k, 0.05 * k))
    _check(vg, orc, ctx, chains, (70,))
