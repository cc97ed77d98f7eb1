"""Batches of several kernel groups, whose passes share a sweep block on two
streams: every chain evolves as in a batch of its own, launched and replayed
from captured blocks several times with other work between."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kinds", [("sc", "bcc"), ("sc", "bcc", "fcc")])
@pytest.mark.parametrize("graph", [False, True])
def test_groups_side_by_side(vg, ctx, kinds, graph):
    K = {"sc": vg.SC, "bcc": vg.BCC, "fcc": vg.FCC}
    H = vg.hamiltonian(exchange=1.0, zeeman=True)
    specs = [(k, d, s) for k in kinds for d, s in (((34, 26, 24), vg.ISING), ((26, 22, 20), vg.HEISENBERG),
                                                   ((6, 4, 4), vg.ISING_BITS))]
    descs = [vg.chain(vg.lattice(K[k], *d), s, vg.RANDOM if i % 2 else vg.FLIP, H, 300 + i)
             for i, (k, d, s) in enumerate(specs)]

    def start(b, i):
        b.set_thermostat(i, 2.5, 0.1)

    want = []
    for d in descs:
        with vg.Batch(ctx, [d]) as b:
            b.randomize()
            start(b, 0)
            sums = b.run_sums(36)[0]
            state = b.get_heisenberg(0) if d.spin == vg.HEISENBERG else b.get_ising(0)
            want.append((sums, state))
    with vg.Batch(ctx, descs) as b:
        b.randomize()
        for i in range(len(descs)):
            start(b, i)
        b.set_graph(graph)
        got = []
        for _ in range(6):
            got.append(b.run_sums(6))
            b.get_ising(0)
        got = [np.concatenate([g[i] for g in got]) for i in range(len(descs))]
        for i, d in enumerate(descs):
            state = b.get_heisenberg(i) if d.spin == vg.HEISENBERG else b.get_ising(i)
            assert np.array_equal(got[i], want[i][0]), i
            assert np.array_equal(state, want[i][1]), i
