"""Matrix chains at two more edges, against the CPU oracle: complete graphs, a
colour a site, of 88 to 92 and of 167 to 170 sites (the descriptor holds the starts
of 168 classes), and rows all of one, two and three entries."""
import numpy as np
import pytest

from test_gpu_graph_rows import _complete

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [88, 92, 167, 168, 169, 170])
def test_colours_around_the_descriptor(vg, orc, ctx, n):
    m = _complete(np.random.default_rng(n), n)
    d = vg.chain(vg.graph_lattice(), vg.ISING, vg.FLIP, vg.hamiltonian(exchange=1.0), 3)
    OM = orc.model(terms=("exchange",), temperature=1.4)
    with vg.Batch(ctx, [d], exchange=[m]) as b:
        b.randomize()
        b.set_thermostat(0, 1.4)
        assert b.colours(0) == n
        G = orc.Graph(*m)
        st = G.ising_init(3)
        assert np.array_equal(b.run_sums(5)[0], G.ising_sweeps(OM, 3, 0, 5, st))
        assert np.array_equal(b.get_ising(0), st)


@pytest.mark.parametrize("proposal", ["flip", "random"])
@pytest.mark.parametrize("spin", ["ising", "heisenberg"])
@pytest.mark.parametrize("n,entries", [(2, 1), (600, 1), (601, 2), (600, 3)])
def test_short_rows(vg, orc, ctx, n, entries, spin, proposal):
    rng = np.random.default_rng(entries)
    i = np.arange(n)
    col = {1: [i ^ 1], 2: [(i + 1) % n, (i - 1) % n],
           3: [i ^ 1, (i + 2) % n, (i - 2) % n]}[entries]
    m = (np.arange(n + 1, dtype=np.uint64) * np.uint64(entries),
         np.stack(col, axis=1).reshape(-1).astype(np.uint64), rng.normal(size=n * entries))
    d = vg.chain(vg.graph_lattice(), vg.ISING if spin == "ising" else vg.HEISENBERG,
                 vg.FLIP if proposal == "flip" else vg.RANDOM, vg.hamiltonian(exchange=1.0), 8)
    OM = orc.model(spin=spin, proposal=proposal, terms=("exchange",), temperature=1.2)
    with vg.Batch(ctx, [d], exchange=[m]) as b:
        b.randomize()
        b.set_thermostat(0, 1.2)
        G = orc.Graph(*m)
        st = G.ising_init(8) if spin == "ising" else G.heis_init(8)
        run = G.ising_sweeps if spin == "ising" else G.heis_sweeps
        assert np.array_equal(b.run_sums(9)[0], run(OM, 8, 0, 9, st))
        end = b.get_ising(0) if spin == "ising" else b.get_heisenberg(0)
        assert np.array_equal(end, st.astype(end.dtype))
