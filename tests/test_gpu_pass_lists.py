"""The edge lists of the Ising tests through the colour passes as well: chains of
that size run in the resident kernel unless a tile is set.  Ferromagnets with the
finest and the coarsest tile, antiferromagnets also in the resident kernel; bit
for bit against the CPU oracle."""
import numpy as np
import pytest

import test_gpu_bcc
import test_gpu_bits
import test_gpu_fcc
import test_gpu_ising

pytestmark = pytest.mark.gpu


def _lists():
    for dims, pbc, T, h, hdir, proposal, terms in test_gpu_ising.CASES:
        yield "sc", dims, pbc, T, h, hdir, proposal, terms
    for dims, pbc, T, h, proposal, terms in test_gpu_bits.CASES[1:]:
        yield "sc", dims, pbc, T, abs(h), (0, 0, 1 if h >= 0 else -1), proposal, terms
    for kind, cases in (("bcc", test_gpu_bcc.ISING), ("fcc", test_gpu_fcc.ISING)):
        for dims, pbc, T, h, hz, proposal, terms in cases:
            yield kind, dims, pbc, T, h, (0, 0, hz), proposal, terms


@pytest.mark.parametrize("exchange", [1.0, -1.0])
@pytest.mark.parametrize("kind,dims,pbc,T,h,hdir,proposal,terms", list(_lists()))
def test_edge_lists_through_the_passes(vg, orc, ctx, kind, dims, pbc, T, h, hdir, proposal, terms,
                                       exchange):
    J = exchange if "exchange" in terms else 0.0
    hdir = tuple(float(v) for v in hdir)
    L = vg.lattice(getattr(vg, kind.upper()), *dims, pbc=tuple(bool(p) for p in pbc))
    H = vg.hamiltonian(exchange=J if "exchange" in terms else None, zeeman="zeeman" in terms)
    d = vg.chain(L, vg.ISING, vg.FLIP if proposal == "flip" else vg.RANDOM, H, 61)
    OL = orc.lattice(kind, *dims, pbc=pbc)
    OM = orc.model(proposal=proposal, terms=terms, exchange=J, temperature=T, field=h,
                   field_dir=hdir)
    start = orc.ising_init(OL, 61)
    want, end = [], start.copy()
    for k, n in enumerate((1, 6)):
        want.append(orc.ising_sweeps(OL, OM, 61, k, n, end))
    for tile in (1, 8) if exchange > 0 else (None, 1, 8):
        with vg.Batch(ctx, [d]) as b:
            if tile:
                b.set_tile(tile)
            b.set_ising(0, start)
            b.set_thermostat(0, T, h, hdir)
            for k, n in enumerate((1, 6)):
                assert np.array_equal(b.run_sums(n)[0], want[k]), (tile, n)
            assert np.array_equal(b.get_ising(0), end), tile
