"""States up and down through the batch's pinned buffer and, past its size, by
copies; refused spins by index; sums of blocks whose records come by copy and
straight to the host."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(2, 1, 1), (30, 20, 10), (170, 170, 150)])  # the last past 4 MiB
def test_ising_states(vg, ctx, dims):
    n = dims[0] * dims[1] * dims[2]
    st = np.random.default_rng(5).choice(np.array([-1, 1], dtype=np.int8), n)
    d = vg.chain(vg.lattice(vg.SC, *dims, pbc=(False,) * 3), vg.ISING, vg.FLIP,
                 vg.hamiltonian(exchange=1.0), 3)
    with vg.Batch(ctx, [d]) as b:
        for s in (st, -st):
            b.set_ising(0, s)
            assert np.array_equal(b.get_ising(0), s)
        for at in (0, n // 2, n - 1):
            bad = st.copy()
            bad[at] = 0
            with pytest.raises(vg.VegasError, match=f"spin {at} is 0"):
                b.set_ising(0, bad)
        assert np.array_equal(b.get_ising(0), -st)


@pytest.mark.parametrize("dims", [(2, 1, 1), (12, 10, 8), (60, 60, 50)])  # the last past 4 MiB
def test_heisenberg_states(vg, ctx, dims):
    n = dims[0] * dims[1] * dims[2]
    v = np.random.default_rng(6).normal(size=(n, 3))
    v = (v / np.linalg.norm(v, axis=1)[:, None]).astype(np.float32).astype(np.float64)
    d = vg.chain(vg.lattice(vg.SC, *dims, pbc=(False,) * 3), vg.HEISENBERG, vg.RANDOM,
                 vg.hamiltonian(exchange=1.0), 3)
    with vg.Batch(ctx, [d]) as b:
        for s in (v, -v):
            b.set_heisenberg(0, s)
            assert np.array_equal(b.get_heisenberg(0), s)


def test_states_from_several_threads(vg, ctx):
    chains = [vg.chain(vg.lattice(vg.SC, 8, 6, 4), vg.ISING, vg.FLIP, vg.hamiltonian(exchange=1.0), k)
              for k in range(8)]
    with vg.Batch(ctx, chains) as b:
        b.randomize()
        want = [b.get_ising(k) for k in range(8)]
        same = [False] * 8

        def read(k):
            same[k] = all(np.array_equal(b.get_ising(k), want[k]) for _ in range(50))

        threads = [threading.Thread(target=read, args=(k,)) for k in range(8)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert all(same)


@pytest.mark.parametrize("chains,dims", [(1, (6, 4, 4)), (40, (4, 4, 2)), (2, (66, 34, 32))])
def test_records_of_long_and_short_runs(vg, orc, ctx, chains, dims):
    ds = [vg.chain(vg.lattice(vg.SC, *dims), vg.ISING, vg.FLIP, vg.hamiltonian(exchange=1.0), 70 + k)
          for k in range(chains)]
    OL = orc.lattice("sc", *dims)
    OM = orc.model(terms=("exchange",), temperature=4.0)
    with vg.Batch(ctx, ds) as b:
        b.randomize()
        for k in range(chains):
            b.set_thermostat(k, 4.0)
        got = [b.run_sums(n) for n in (1, 30, 2)]
        for k in range(chains):
            st = orc.ising_init(OL, 70 + k)
            want = orc.ising_sweeps(OL, OM, 70 + k, 0, 33, st)
            assert np.array_equal(np.concatenate([g[k] for g in got]), want), k
