"""Matrix chains at the edges of their passes, on the GPU vs the CPU oracle bit
for bit: rows of the same length around the entries gathered at once (8) and
rows of different lengths with empty ones, one chain alone and two in a batch,
more colours than the descriptor holds class starts for, and couplings whose
bond sums take all 64 bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ring(rng, n, reach, scale=1.0):
    """Site i coupled to i +- 1 .. i +- reach: 2 * reach entries in every row."""
    col = [[(i + s * d) % n for d in range(1, reach + 1) for s in (1, -1)] for i in range(n)]
    val = rng.normal(size=(n, 2 * reach)) * scale
    return (np.arange(n + 1, dtype=np.uint64) * np.uint64(2 * reach),
            np.array(col, dtype=np.uint64).reshape(-1), val.reshape(-1))


def _uneven(rng, n):
    rows = [sorted(set(int(j) for j in rng.integers(0, n, size=rng.integers(0, 20))) - {i})
            if i % 5 else [] for i in range(n)]
    ptr = np.cumsum([0] + [len(r) for r in rows])
    col = np.array([j for r in rows for j in r], dtype=np.uint64)
    return ptr.astype(np.uint64), col, rng.normal(size=len(col))


def _complete(rng, n):
    col = [[j for j in range(n) if j != i] for i in range(n)]
    return (np.arange(n + 1, dtype=np.uint64) * np.uint64(n - 1),
            np.array(col, dtype=np.uint64).reshape(-1), rng.normal(size=n * (n - 1)) / np.sqrt(n))


def _matrices():
    rng = np.random.default_rng(19)
    return {"ring 6": [_ring(rng, 700, 3)], "ring 8": [_ring(rng, 130, 4)],
            "ring 10": [_ring(rng, 65, 5)], "ring 18": [_ring(rng, 257, 9)],
            "uneven": [_uneven(rng, 333)], "complete 180": [_complete(rng, 180)],
            "two chains": [_ring(rng, 300, 2), _uneven(rng, 90)],
            "large couplings": [_ring(rng, 200, 3, 1e6)]}


@pytest.mark.parametrize("spin,proposal", [("ising", "flip"), ("ising", "random"),
                                           ("heisenberg", "random"), ("heisenberg", "flip")])
@pytest.mark.parametrize("name", list(_matrices()))
def test_graph_rows(vg, orc, ctx, name, spin, proposal):
    mats = _matrices()[name]
    H = vg.hamiltonian(exchange=1.0, zeeman=True)
    descs = [vg.chain(vg.graph_lattice(), vg.ISING if spin == "ising" else vg.HEISENBERG,
                      vg.FLIP if proposal == "flip" else vg.RANDOM, H, 40 + k)
             for k in range(len(mats))]
    OM = orc.model(spin=spin, proposal=proposal, terms=("exchange", "zeeman"), temperature=1.4,
                   field=0.2)
    with vg.Batch(ctx, descs, exchange=mats) as b:
        b.randomize()
        for k in range(len(mats)):
            b.set_thermostat(k, 1.4, 0.2)
        got = b.run_sums(12)
        for k, m in enumerate(mats):
            G = orc.Graph(*m)
            st = G.ising_init(40 + k) if spin == "ising" else G.heis_init(40 + k)
            run = G.ising_sweeps if spin == "ising" else G.heis_sweeps
            assert np.array_equal(got[k], run(OM, 40 + k, 0, 12, st)), k
            end = b.get_ising(k) if spin == "ising" else b.get_heisenberg(k)
            assert np.array_equal(end, st.astype(end.dtype)), k
