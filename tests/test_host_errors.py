"""What the engine's host code leaves behind when a HIP call fails part way: on the
stand-in for the HIP runtime."""
import pytest

import _fake


@pytest.mark.parametrize("failing", [1, 2, 3, 5, 7])
def test_noalloc_unpacks_after_an_error(failing):
    """int8 planes packed in place are unpacked again when a launch of the sweeps
    (3, 5) or their reduction (7) fails, and left alone when the set-up or the
    packing itself (1, 2) does."""
    out = _fake.run(f"""
d = sc(800)
fake.fake_error_at_launch({failing})
try:
    vg.run_sums_noalloc(d, 4.5, 0.0, (0.0, 0.0, 1.0), 0, 2, 4096, 8192, 0)
except vg.VegasError:
    print("refused")
print(launches()[-1])
""")
    assert out.startswith("refused")
    last = out.split()[-1]
    assert ("noalloc_bitsILb0E" in last) == (failing > 2), last
    if failing <= 2:
        assert ("noalloc_setup", "noalloc_bitsILb1E")[failing - 1] in last, last


def test_noalloc_enqueues_nothing_after_an_older_error():
    """An error that an earlier call left behind fails the call before it has
    touched the caller's planes."""
    out = _fake.run("""
fake.fake_fail(b"hipMalloc", 1)
p = C.c_void_p()
assert fake.hipMalloc(C.byref(p), C.c_size_t(16)) != 0
try:
    vg.run_sums_noalloc(sc(800), 4.5, 0.0, (0.0, 0.0, 1.0), 0, 2, 4096, 8192, 0)
except vg.VegasError:
    print("refused")
print(len(launches()))
""")
    assert out.split() == ["refused", "0"]


@pytest.mark.parametrize("sweeps,failing", [(2, 1), (2, 3), (2, 6), (5000, 3), (5000, 8194)])
def test_noalloc_writes_bytes_after_an_error(sweeps, failing):
    """The same of a chain whose bits are held apart: its bytes are written after
    a failure behind the packing, in the first chunk of sweeps (4096) and later."""
    out = _fake.run(f"""
fake.fake_error_at_launch({failing})
try:
    vg.run_sums_noalloc(sc(32), 4.5, 0.0, (0.0, 0.0, 1.0), 0, {sweeps}, 4096, 8192, 0)
except vg.VegasError:
    print("refused")
l = launches()
print(len(l), l[-1])
""")
    assert out.startswith("refused")
    count, last = out.split()[1:]
    if failing == 1:
        assert count == "1"
    else:
        assert "noalloc_finish" in last, last


TWO_GROUPS = """
b = vg.Batch(ctx, [sc(64), sc(64, spin=vg.HEISENBERG)])
b.run(1)
fake.fake_clear()
"""


@pytest.mark.parametrize("how,last", [
    ("fake_error_at_launch(3)", "wait"), ("fake_error_at_launch(7)", "wait"),
    ('fake_fail(b"hipEventRecord", 3)', "sync"), ('fake_fail(b"hipStreamWaitEvent", 2)', "sync"),
])
def test_side_stream_joins_after_an_error(how, last):
    """A block of two groups whose launch fails: whatever the second stream was
    given lies before the next work of the main stream, by its event or, if that
    fails, by waiting."""
    out = _fake.run(TWO_GROUPS + f"""
fake.{how}
try:
    b.run(1)
except vg.VegasError:
    print("refused")
print(";".join(log()))
""")
    refused, lines = out.strip().split("\n")
    assert refused == "refused"
    lines = lines.split(";")
    streams = [l.split()[l.split().index("stream") + 1] for l in lines if l.startswith("launch")]
    main = streams[0]
    side = next(s for s in streams if s != main)
    tail = lines[max(i for i, l in enumerate(lines) if f"stream {side} " in l and "launch" in l) + 1:]
    if last == "wait":
        assert any(l.startswith("record event") and l.endswith(f"stream {side}") for l in tail), tail
        assert any(l.startswith(f"wait stream {main} ") for l in tail), tail
    else:
        assert f"sync stream {side}" in tail, tail


@pytest.mark.parametrize("spin,call", [
    ("ISING", "set_ising(0, [1] * 64)"), ("ISING", "get_ising(0)"),
    ("HEISENBERG", "set_heisenberg(0, [[0.0, 0.0, 1.0]] * 64)"), ("HEISENBERG", "get_heisenberg(0)"),
])
def test_state_buffer_is_waited_for_after_an_error(spin, call):
    """A kernel that reads or writes the pinned state buffer has ended before the
    call returns an error: the next call writes there."""
    out = _fake.run(f"""
b = vg.Batch(ctx, [sc(4, spin=vg.{spin})])
fake.fake_clear()
fake.fake_error_at_launch(1)
try:
    b.{call}
except vg.VegasError:
    print("refused")
print(";".join(log()))
""")
    refused, lines = out.strip().split("\n")
    assert refused == "refused"
    lines = lines.split(";")
    assert any(l.startswith("launch") for l in lines), lines
    assert lines[-1].startswith("sync stream"), lines


@pytest.mark.parametrize("failing,of_server", [("hipStreamCreateWithFlags", 2),
                                               ("hipEventCreateWithFlags", 1)])
def test_one_stream_where_a_second_cannot_be_made(failing, of_server):
    """Batches and servers with chains of two groups run on one stream then."""
    out = _fake.run(f"""
fake.fake_fail(b"{failing}", 1)
b = vg.Batch(ctx, [sc(64), sc(64, spin=vg.HEISENBERG)])
b.run(1)
s1 = {{l.split()[3] for l in log() if l.startswith("launch")}}
fake.fake_fail(b"{failing}", {of_server})  # (the server's first stream is made before)
s = vg.Server(ctx, quantum_sweeps=10)
fake.fake_clear()
ids = [s.submit(sc(64, spin=k), vg.relax(10, 2.0)) for k in (vg.ISING, vg.HEISENBERG)]
states = [s.wait(j).state for j in ids]
s2 = {{l.split()[3] for l in log() if l.startswith("launch")}}
print(len(s1), len(s2), states == [vg.JOB_DONE] * 2)
""")
    assert out.split() == ["1", "1", "True"]
