"""The multispin Ising passes at the edges of their words and plans, on the GPU
vs the CPU oracle bit for bit: row lengths around a word of 32 positions, every
tile with a remainder, chains with and without a field (general and plain
acceptance plans) and with open ends (words whose sites differ in their absent
neighbours); and the allocation-free sweeps on rows of one byte per site,
whose bits are packed in place and unpacked again."""
import numpy as np
import pytest

from test_zz_no_alloc import _Hip, _from_planes, _to_planes

pytestmark = pytest.mark.gpu

KINDS = {"sc": 0, "bcc": 1, "fcc": 2}
T = {"sc": 4.5, "bcc": 6.3, "fcc": 9.8}


def _chain(vg, orc, kind, w, ly, lz, pbc, field, seed, spin="int8", proposal="flip"):
    dims = (2 * w if kind == "sc" else w, ly, lz)
    L = vg.lattice([vg.SC, vg.BCC, vg.FCC][KINDS[kind]], *dims, pbc=tuple(bool(p) for p in pbc))
    d = vg.chain(L, vg.ISING_BITS if spin == "bits" else vg.ISING,
                 vg.RANDOM if proposal == "random" else vg.FLIP,
                 vg.hamiltonian(exchange=1.0, zeeman=True), seed)
    OL = orc.lattice(kind, *dims, pbc=pbc)
    OM = orc.model(proposal=proposal, terms=("exchange", "zeeman"), temperature=T[kind], field=field)
    return L, d, OL, OM


@pytest.mark.parametrize("kind", ["sc", "bcc", "fcc"])
@pytest.mark.parametrize("w,ly,lz,pbc", [
    (1, 4, 10, (1, 1, 1)), (16, 2, 2, (1, 1, 1)), (31, 4, 6, (1, 1, 1)), (32, 6, 10, (1, 1, 1)),
    (33, 4, 18, (1, 1, 1)), (65, 2, 6, (1, 1, 1)),
    (31, 5, 7, (0, 0, 0)), (32, 3, 9, (0, 0, 1)), (33, 5, 3, (0, 1, 0)), (64, 3, 5, (1, 0, 0)),
])
def test_words_plans_and_tiles(vg, orc, ctx, kind, w, ly, lz, pbc):
    if kind == "sc" and pbc[1]:
        ly += ly & 1
    if kind == "sc" and pbc[2]:
        lz += lz & 1
    for k, (field, proposal, spin) in enumerate([(0.0, "flip", "int8"), (0.3, "flip", "bits"),
                                                 (0.3, "random", "int8")]):
        L, d, OL, OM = _chain(vg, orc, kind, w, ly, lz, pbc, field, 61 + k, spin, proposal)
        st = orc.ising_init(OL, 61 + k)
        with vg.Batch(ctx, [d]) as b:
            b.randomize()
            b.set_thermostat(0, T[kind], field)
            step = 0
            for tile in (0, 1, 2, 4, 8):  # 0: the tile the batch starts with
                if tile:
                    b.set_tile(tile)
                want = orc.ising_sweeps(OL, OM, 61 + k, step, 3, st)
                assert np.array_equal(b.run_sums(3)[0], want), (field, proposal, tile)
                assert np.array_equal(b.get_ising(0), st), (field, proposal, tile)
                step += 3


@pytest.mark.parametrize("kind,w,ly,lz,pbc", [
    ("sc", 8, 4, 2, (1, 1, 1)), ("sc", 13, 5, 1, (1, 0, 0)),       # 64 (one wave) and 65 sites a colour
    ("sc", 32, 8, 4, (1, 1, 1)), ("bcc", 41, 5, 5, (0, 1, 0)),     # 1024 and 1025: 1 and 2 a lane
    ("sc", 33, 8, 8, (1, 1, 1)), ("bcc", 16, 16, 8, (1, 1, 1)),    # 2112 and 2048: 4 and 2 a lane
    ("sc", 64, 8, 8, (1, 1, 1)), ("bcc", 17, 15, 16, (0, 0, 1)),   # 4096 and 4080: the largest
    ("fcc", 32, 8, 8, (1, 1, 0)), ("fcc", 1, 1, 1, (1, 1, 1)),     # 2048, the largest of fcc, and 1
    ("fcc", 9, 5, 23, (1, 0, 1)),                                  # 1035
])
def test_resident_chains_equal_passes(vg, orc, ctx, kind, w, ly, lz, pbc):
    """Sweep blocks in one workgroup against colour passes (a set tile) and the
    oracle, batches of two fields and both proposals, over two blocks and the
    seams of the batches of draws."""
    chains = [_chain(vg, orc, kind, w, ly, lz, pbc, f, 81 + k, p, q)
              for k, (f, p, q) in enumerate([(0.0, "int8", "flip"), (0.4, "bits", "random"),
                                             (-0.2, "int8", "flip")])]
    states = [orc.ising_init(c[2], 81 + k) for k, c in enumerate(chains)]
    want = [orc.ising_sweeps(c[2], c[3], 81 + k, 0, 300, s)
            for k, (c, s) in enumerate(zip(chains, states))]
    for tile in (0, 1):
        with vg.Batch(ctx, [c[1] for c in chains]) as b:
            b.randomize()
            for k, f in enumerate((0.0, 0.4, -0.2)):
                b.set_thermostat(k, T[kind], f)
            if tile:
                b.set_tile(tile)
            got = b.run_sums(300)
            for k in range(3):
                assert np.array_equal(got[k], want[k]), (tile, k)
                assert np.array_equal(b.get_ising(k), states[k]), (tile, k)


@pytest.mark.parametrize("kind,w,ly,lz,pbc,field", [
    ("bcc", 7, 5, 9, (1, 1, 1), 0.0),        # an odd number of rows
    ("fcc", 33, 5, 4, (0, 1, 0), 0.2),
    ("sc", 1, 2, 4, (1, 1, 1), 0.0),
    ("sc", 2080, 2, 2, (1, 1, 1), 0.1),      # rows of 65 words: two chunks of a wave
    ("bcc", 4100, 1, 3, (1, 0, 1), 0.0),     # three chunks, the last of one word
])
def test_noalloc_packs_and_unpacks_byte_rows(vg, orc, ctx, kind, w, ly, lz, pbc, field):
    hip = _Hip()
    L, d, OL, OM = _chain(vg, orc, kind, w, ly, lz, pbc, field, 71)
    st = orc.ising_init(OL, 71)
    planes = _to_planes(L, False, st)
    init = np.zeros((4, 5), dtype=np.int64)
    spins, sums = hip.upload(planes), hip.upload(init)
    try:
        vg.run_sums_noalloc(d, T[kind], field, (0.0, 0.0, 1.0), 2, 4, spins, sums, 0)
        hip.sync()
        got, out = hip.download(sums, init), hip.download(spins, planes)
    finally:
        hip.free(spins)
        hip.free(sums)
    want = orc.ising_sweeps(OL, OM, 71, 2, 4, st)
    assert np.array_equal(got[:, :4], want[:, :4])
    assert np.array_equal(_from_planes(L, False, out), st)
    assert np.array_equal(out, _to_planes(L, False, st))  # padding zero again


@pytest.mark.parametrize("ly,lz", [(512, 512), (512, 514)])  # 1024 and 1028 workgroups of short rows
def test_sums_of_many_workgroups(vg, orc, ctx, ly, lz):
    L, d, OL, OM = _chain(vg, orc, "sc", 1, ly, lz, (1, 1, 1), 0.0, 91)
    st = orc.ising_init(OL, 91)
    with vg.Batch(ctx, [d]) as b:
        b.randomize()
        b.set_thermostat(0, T["sc"])
        b.set_tile(1)
        assert np.array_equal(b.run_sums(3)[0], orc.ising_sweeps(OL, OM, 91, 0, 3, st))
