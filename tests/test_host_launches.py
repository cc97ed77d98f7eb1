"""What the engine's host code asks of the HIP runtime, and when: on the stand-in
for it."""
import pytest

import _fake


@pytest.mark.parametrize("spin", ["ISING", "HEISENBERG"])
def test_state_buffer_is_made_with_the_batch(spin):
    """The first download and upload allocate nothing; nor does a chain of another
    size in the batch."""
    out = _fake.run(f"""
b = vg.Batch(ctx, [sc(8, spin=vg.{spin}), sc(20, spin=vg.{spin})])
fake.fake_clear()
if vg.{spin} == vg.ISING:
    import numpy as np
    b.set_ising(0, np.ones(512, dtype=np.int8)); b.set_ising(1, np.ones(8000, dtype=np.int8))
    b.get_ising(0); b.get_ising(1)
else:
    b.set_heisenberg(0, [[0.0, 0.0, 1.0]] * 512); b.set_heisenberg(1, [[0.0, 0.0, 1.0]] * 8000)
    b.get_heisenberg(0); b.get_heisenberg(1)
print(sum(l.startswith("hostmalloc") for l in log()), sum(l.startswith("copy") for l in log()))
""")
    assert out.split() == ["0", "0"]


def test_batch_without_a_state_buffer():
    """Where the pinned memory for it cannot be had, states are copied."""
    out = _fake.run("""
fake.fake_fail(b"hipHostMalloc", 3)   # (after the two of the group's descriptors)
b = vg.Batch(ctx, [sc(8)])
fake.fake_clear()
import numpy as np
b.set_ising(0, np.ones(512, dtype=np.int8))
b.run(2)
print(sum(l.startswith("copy") for l in log()))
""")
    assert out.split() == ["1"]


def test_server_makes_its_streams_at_creation():
    out = _fake.run("""
s = vg.Server(ctx, quantum_sweeps=10)
fake.fake_clear()
ids = [s.submit(sc(64, spin=k), vg.relax(10, 2.0)) for k in (vg.ISING, vg.HEISENBERG)]
for j in ids: s.wait(j)
s.close()
print(sum(l.startswith("stream") for l in log()),
      len({l.split()[3] for l in log() if l.startswith("launch")}))
""")
    assert out.split() == ["0", "2"]


@pytest.mark.parametrize("change", ["set_tile(2)", "set_tie_capacity(3)"])
def test_second_stream_for_groups_that_turn_to_passes(change):
    """Small chains of two lattices run a block in one launch each; made to run
    passes, they do so side by side."""
    out = _fake.run(f"""
b = vg.Batch(ctx, [sc(8), sc(8, kind=vg.BCC)])
b.run(2)
one = {{l.split()[3] for l in log() if l.startswith("launch")}}
b.{change}
fake.fake_clear()
b.run(2)
print(len(one), len({{l.split()[3] for l in log() if "_pass" in l}}))
""")
    assert out.split() == ["1", "2"]


def test_draws_take_no_memory_from_the_rest():
    """A batch that fits without the workspace for the draws of its small Heisenberg
    chains is made, and runs passes: here one byte short of all."""
    out = _fake.run("""
descs = [sc(16, spin=vg.HEISENBERG, seed=k) for k in range(4)]
descs.append(sc(16, proposal=vg.WOLFF))
before = fake.fake_used()
b = vg.Batch(ctx, descs)
used = fake.fake_used() - before
b.run(2)
print(any("heis_draws" in l for l in launches()))
b.close()
fake.fake_limit(fake.fake_used() + used - 1)
b = vg.Batch(ctx, descs)
fake.fake_clear()
b.run(2)
print(any("heis_draws" in l for l in launches()), any("heis_sc_pass" in l for l in launches()))
""")
    assert out.split() == ["True", "False", "True"]


def test_blocks_send_sweep_counters_only():
    """Descriptors go to the device when something but the sweep counters has
    changed: a thermostat, a tile."""
    out = _fake.run("""
b = vg.Batch(ctx, [sc(4, seed=k) for k in range(2000)])
def sent(n):
    fake.fake_clear()
    b.run(n)
    most = max(int(l.split()[-1]) for l in log() if l.startswith("copy"))
    return int(most > 2000 * n * 40), sum("set_sweeps" in l for l in launches())
print(*sent(1), *sent(1), *sent(2), *sent(300))
b.set_thermostat(7, 2.0)
print(*sent(1), *sent(1))
b.set_tile(2)
print(*sent(1), *sent(1))
b.set_sweep_count(3, 77)
print(*sent(1))
""")
    # (descriptors sent, launches for counters)
    assert out.split("\n")[:4] == ["0 0 0 1 0 1 0 2", "1 0 0 1", "1 0 0 1", "0 1"]
