"""The allocation-free sweeps' conversion of int8 planes: in the scratch, at the
edges of a workgroup's share (1024 sixteens of positions a colour, 4096 after many
workgroups' sums) and over more sweeps than one chunk holds, against the oracle;
in place, for a chain too large for the scratch, against the bit-packed call."""
import numpy as np
import pytest

from test_gpu_multispin import T, _chain
from test_zz_no_alloc import _Hip, _from_planes, _to_planes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,w,ly,lz,sweeps", [
    ("sc", 16, 2, 2, 1), ("sc", 17, 2, 4, 2),
    ("sc", 32, 16, 32, 1),     # 1024 sixteens a colour
    ("bcc", 48, 19, 27, 3),    # 2052: four more than two workgroups'; pitch past the words
    ("fcc", 70, 13, 10, 2),
    ("sc", 1, 512, 514, 2),    # 1028 workgroups: sums by 1024 threads
    ("bcc", 5, 4, 3, 4097),    # two chunks
])
def test_noalloc_converts_in_the_scratch(vg, orc, ctx, kind, w, ly, lz, sweeps):
    hip = _Hip()
    L, d, OL, OM = _chain(vg, orc, kind, w, ly, lz, (1, 1, 1), 0.0, 23)
    st = orc.ising_init(OL, 23)
    planes = _to_planes(L, False, st)
    init = np.zeros((sweeps, 5), dtype=np.int64)
    spins, sums = hip.upload(planes), hip.upload(init)
    try:
        vg.run_sums_noalloc(d, T[kind], 0.0, (0.0, 0.0, 1.0), 5, sweeps, spins, sums, 0)
        hip.sync()
        got, out = hip.download(sums, init), hip.download(spins, planes)
    finally:
        hip.free(spins)
        hip.free(sums)
    want = orc.ising_sweeps(OL, OM, 23, 5, sweeps, st)
    assert np.array_equal(got[:, :4], want[:, :4])
    assert np.array_equal(_from_planes(L, False, out), st)
    assert np.array_equal(out, _to_planes(L, False, st))  # padding stays zero


def test_noalloc_converts_in_place(vg, ctx):
    """321 million sites: 42 million bytes of bits, rows of 65 words."""
    hip = _Hip()
    w, ly, lz, sweeps = 2080, 280, 276, 3
    L = vg.lattice(vg.SC, 2 * w, ly, lz)
    ham = vg.hamiltonian(exchange=1.0)
    rows, pitch, bpitch = ly * lz, 2112, 272
    outs, recs = [], []
    for spin in (vg.ISING, vg.ISING_BITS):
        if spin == vg.ISING:
            one = np.zeros(pitch, dtype=np.uint8)
            one[:w] = 1
        else:
            one = np.zeros(bpitch, dtype=np.uint8)
            one[:w // 8] = 255
        plane = (rows * len(one) + 255) // 256 * 256
        planes = np.zeros((2, plane), dtype=np.uint8)
        planes[:, :rows * len(one)] = np.tile(one, rows)
        init = np.zeros((sweeps, 5), dtype=np.int64)
        spins, sums = hip.upload(planes), hip.upload(init)
        try:
            vg.run_sums_noalloc(vg.chain(L, spin, vg.FLIP, ham, 3), 4.5, 0.0, (0.0, 0.0, 1.0), 0,
                                sweeps, spins, sums, 0)
            hip.sync()
            recs.append(hip.download(sums, init))
            outs.append(hip.download(spins, planes)[:, :rows * len(one)].reshape(2, rows, len(one)))
        finally:
            hip.free(spins)
            hip.free(sums)
    assert np.array_equal(recs[0], recs[1])
    assert not outs[0][:, :, w:].any()
    for c in range(2):
        bits = np.unpackbits(outs[1][c][:, :w // 8], axis=1, bitorder="little")
        assert np.array_equal(outs[0][c][:, :w], bits), c
