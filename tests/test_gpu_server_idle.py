"""What a Heisenberg job that sits a quantum out costs the jobs that run: less
than half of what moving its spins once would take."""
import pytest

pytestmark = pytest.mark.gpu

SWEEPS = 200


def _device_ms(vg, ctx, kind, dims, beside):
    ham = vg.hamiltonian(exchange=1.0)
    small = vg.chain(vg.lattice(kind, 24, 24, 24), vg.HEISENBERG, vg.RANDOM, ham, 1)
    # every quantum's budget is one site's work: the first job runs alone
    with vg.Server(ctx, memory_bytes=1 << 30, quantum_sweeps=100, sweep_budget=1) as s:
        ids = [s.submit(small, vg.relax(SWEEPS, 1.2))]
        if beside:
            big = vg.chain(vg.lattice(kind, *dims), vg.HEISENBERG, vg.RANDOM, ham, 2)
            ids.append(s.submit(big, vg.relax(1, 1.2)))
        for j in ids:
            s.wait(j)
        return s.stats().device_ms


@pytest.mark.parametrize("kind,dims", [("SC", (256, 256, 256)), ("BCC", (200, 200, 200)),
                                       ("FCC", (160, 160, 160))])
def test_idle_heisenberg_job(vg, ctx, kind, dims):
    kind = getattr(vg, kind)
    _device_ms(vg, ctx, kind, dims, True)  # first launches
    alone = min(_device_ms(vg, ctx, kind, dims, False) for _ in range(2))
    beside = min(_device_ms(vg, ctx, kind, dims, True) for _ in range(2))
    # a sweep reads and writes 12 bytes a site, at 8 TB/s at best; the job's own
    # sweep and the launches of its passes are within the other half
    sites = dims[0] * dims[1] * dims[2] * {vg.SC: 1, vg.BCC: 2, vg.FCC: 4}[kind]
    bound = 0.5 * SWEEPS * 24 * sites / 8e12 * 1e3
    print(f"alone {alone:.3f} ms, beside {beside:.3f} ms, bound on the difference {bound:.3f} ms")
    assert beside - alone < bound
