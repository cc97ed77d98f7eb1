"""Heisenberg items of four positions on small chains: in a batch with one large
chain, past the line from which a group takes them (8, 14 and 48 waves of single
sites a SIMD on sc, bcc and fcc), chains with rows shorter than an item, rows that
are no multiple of one, and open ends; bit for bit against the CPU oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LARGE = {"sc": (106, 102, 100), "bcc": (99, 98, 97), "fcc": (148, 147, 147)}
SMALL = [
    ((2, 4, 6), (1, 1, 1)), ((4, 6, 2), (0, 1, 1)), ((6, 4, 4), (1, 0, 0)),
    ((10, 5, 3), (0, 0, 0)), ((14, 4, 6), (1, 1, 1)), ((38, 3, 5), (1, 0, 0)),
]
ODD = [((1, 3, 5), (1, 1, 1)), ((3, 5, 2), (0, 1, 0)), ((5, 1, 7), (1, 1, 1)),
       ((7, 3, 3), (0, 0, 1))]


@pytest.mark.parametrize("proposal", ["random", "flip"])
@pytest.mark.parametrize("kind", ["sc", "bcc", "fcc"])
def test_small_chains_with_items_of_four(vg, orc, ctx, kind, proposal):
    terms = ("exchange", "anisotropy", "zeeman")
    ham = vg.hamiltonian(exchange=1.0, anisotropy=0.3, zeeman=True)
    prop = vg.RANDOM if proposal == "random" else vg.FLIP
    cases = SMALL + (ODD if kind != "sc" else [])
    lattice = getattr(vg, kind.upper())
    descs = [vg.chain(vg.lattice(lattice, *LARGE[kind]), vg.HEISENBERG, prop, ham, 5)]
    descs += [vg.chain(vg.lattice(lattice, *dims, pbc=tuple(bool(p) for p in pbc)), vg.HEISENBERG,
                       prop, ham, 70 + k) for k, (dims, pbc) in enumerate(cases)]
    OM = orc.model(spin="heisenberg", proposal=proposal, terms=terms, anisotropy=0.3,
                   temperature=1.1, field=0.2)
    with vg.Batch(ctx, descs) as b:
        b.randomize()
        for k in range(len(descs)):
            b.set_thermostat(k, 1.1, 0.2)
        got = b.run_sums(3)
        for k, (dims, pbc) in enumerate(cases):
            OL = orc.lattice(kind, *dims, pbc=pbc)
            st = orc.heis_init(OL, 70 + k)
            assert np.array_equal(got[1 + k], orc.heis_sweeps(OL, OM, 70 + k, 0, 3, st)), dims
            assert np.array_equal(b.get_heisenberg(1 + k), st.astype(np.float64)), dims

