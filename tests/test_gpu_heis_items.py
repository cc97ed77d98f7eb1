"""Heisenberg colour passes with one and four positions per work item, which the
amount of work chooses: bit-exact against the CPU oracle on lattices past the
resident chains' size whose rows are no multiple of four, with open ends, and on
small chains through the passes (per-pass timing runs them)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KINDS = {"sc": 0, "bcc": 1, "fcc": 2}


def _run(vg, orc, ctx, kind, dims, pbc, proposal, sweeps, timing=False):
    L = vg.lattice([vg.SC, vg.BCC, vg.FCC][KINDS[kind]], *dims, pbc=tuple(bool(p) for p in pbc))
    d = vg.chain(L, vg.HEISENBERG, vg.RANDOM if proposal == "random" else vg.FLIP,
                 vg.hamiltonian(exchange=1.0, anisotropy=-0.3, zeeman=True), 57)
    OL = orc.lattice(kind, *dims, pbc=pbc)
    OM = orc.model(spin="heisenberg", proposal=proposal, terms=("exchange", "anisotropy", "zeeman"),
                   anisotropy=-0.3, temperature=1.2, field=0.15)
    st = orc.heis_init(OL, 57)
    with vg.Batch(ctx, [d]) as b:
        b.randomize()
        b.set_thermostat(0, 1.2, 0.15)
        if timing:
            b.set_timing(True)
        assert np.array_equal(b.run_sums(sweeps)[0], orc.heis_sweeps(OL, OM, 57, 0, sweeps, st))
        assert np.array_equal(b.get_heisenberg(0), st.astype(np.float64))


@pytest.mark.parametrize("proposal", ["random", "flip"])
@pytest.mark.parametrize("kind,dims,pbc", [
    ("sc", (34, 17, 18), (1, 0, 1)), ("sc", (130, 9, 10), (0, 0, 0)),
    ("bcc", (17, 17, 16), (0, 1, 1)), ("bcc", (67, 8, 9), (1, 1, 0)),
    ("fcc", (17, 13, 11), (1, 1, 1)), ("fcc", (9, 19, 14), (0, 0, 1)),
])
def test_single_items(vg, orc, ctx, kind, dims, pbc, proposal):
    _run(vg, orc, ctx, kind, dims, pbc, proposal, 4)


@pytest.mark.parametrize("kind,dims,pbc", [
    ("sc", (106, 102, 98), (1, 1, 1)),    # 8279 waves of single items: past 8 a SIMD
    ("sc", (130, 96, 88), (0, 1, 1)),
    ("bcc", (99, 97, 97), (1, 0, 1)),     # 14554: past 14 a SIMD
])
def test_items_of_four(vg, orc, ctx, kind, dims, pbc):
    for proposal in ("random", "flip"):
        _run(vg, orc, ctx, kind, dims, pbc, proposal, 1)


@pytest.mark.parametrize("kind,dims", [("sc", (6, 5, 7)), ("bcc", (3, 4, 5)), ("fcc", (5, 3, 2))])
def test_small_chains_through_the_passes(vg, orc, ctx, kind, dims):
    for proposal in ("random", "flip"):
        _run(vg, orc, ctx, kind, dims, (0, 0, 0), proposal, 5, timing=True)
