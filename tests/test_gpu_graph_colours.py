"""Matrix chains around the number of colours whose class starts the descriptor
holds (90): complete graphs, a colour a site, against the CPU oracle."""
import numpy as np
import pytest

from test_gpu_graph_rows import _complete

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [88, 89, 90, 91, 92])
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
