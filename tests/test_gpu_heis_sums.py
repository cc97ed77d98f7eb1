"""Sums of small Heisenberg chains whose terms are larger than a unit spin's: a
lane of the resident kernel adds up to eight sites a sweep, each below 16 in every
sum, and their total has to be exact (the oracle's sums are 64-bit)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(vg, orc, ctx, kind, dims, pbc, axis, length, proposal):
    L = vg.lattice({"sc": vg.SC, "bcc": vg.BCC, "fcc": vg.FCC}[kind], *dims,
                   pbc=tuple(bool(p) for p in pbc))
    terms = ("exchange", "anisotropy", "zeeman")
    d = vg.chain(L, vg.HEISENBERG, vg.RANDOM if proposal == "random" else vg.FLIP,
                 vg.hamiltonian(exchange=1.0, anisotropy=-0.5, axis=axis, zeeman=True), 11)
    OL = orc.lattice(kind, *dims, pbc=pbc)
    OM = orc.model(spin="heisenberg", proposal=proposal, terms=terms, anisotropy=-0.5, axis=axis,
                   temperature=0.2, field=0.1)
    st = np.tile(np.array([0.0, 0.0, length], dtype=np.float32), (orc.num_sites(OL), 1))
    with vg.Batch(ctx, [d]) as b:
        b.set_heisenberg(0, st.astype(np.float64))
        b.set_thermostat(0, 0.2, 0.1)
        assert np.array_equal(b.run_sums(3)[0], orc.heis_sweeps(OL, OM, 11, 0, 3, st))
        assert np.array_equal(b.get_heisenberg(0), st.astype(np.float64))


@pytest.mark.parametrize("kind,dims", [
    ("sc", (20, 20, 20)), ("bcc", (16, 16, 16)), ("fcc", (12, 12, 12)),  # eight sites a lane
    ("sc", (16, 16, 16)), ("fcc", (9, 9, 9)),                            # four
    ("sc", (2, 32, 32)),                                                 # two, one site a row
])
@pytest.mark.parametrize("axis", [(0.0, 0.0, 1.7), (0.0, 0.0, 3.9)])
def test_long_anisotropy_axis(vg, orc, ctx, kind, dims, axis):
    _run(vg, orc, ctx, kind, dims, (1, 1, 1), axis, 1.0, "flip")


@pytest.mark.parametrize("proposal", ["flip", "random"])
def test_long_spins(vg, orc, ctx, proposal):
    """Length 2.7: two neighbours keep a site's bonds below 16."""
    _run(vg, orc, ctx, "sc", (8192, 1, 1), (1, 0, 0), (0.0, 0.0, 1.0), 2.7, proposal)


def test_long_spins_under_replays(vg, orc, ctx):
    """A captured block follows the lengths of the spins: unit, long, unit again."""
    L = vg.lattice(vg.SC, 8192, 1, 1, pbc=(True, False, False))
    d = vg.chain(L, vg.HEISENBERG, vg.FLIP, vg.hamiltonian(exchange=1.0), 11)
    OL = orc.lattice("sc", 8192, 1, 1, pbc=(1, 0, 0))
    OM = orc.model(spin="heisenberg", terms=("exchange",), temperature=0.2)
    with vg.Batch(ctx, [d]) as b:
        b.set_graph(True)
        b.set_thermostat(0, 0.2)
        for length in (1.0, 2.7, 1.0):
            b.randomize()
            st = orc.heis_init(OL, 11)
            if length != 1.0:
                st = np.tile(np.array([0.0, 0.0, length], dtype=np.float32), (8192, 1))
                b.set_heisenberg(0, st.astype(np.float64))
            for k in range(2):
                assert np.array_equal(b.run_sums(3)[0],
                                      orc.heis_sweeps(OL, OM, 11, 3 * k, 3, st)), (length, k)
