"""GPU: the graph form's packed mtask kernels (four lanes per thread) where a
group of four lanes is cut: by the lane count, by a block's end, by lanes that
are done or hold another cycle's clock. Whole numbers: exact."""
import numpy as np
import pytest

import oracle
from rtlflow_amd.designs import registry
from rtlflow_amd.model import MODE_FUSED, MODE_GRAPH

SEED = registry.SEED_CFG[2]


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["net_tiny", "net_ram"])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 255, 257, 1026])
def test_packed_graph_lane_counts(gpu, name, n):
    """Hashes and each lane's whole state, graph form against the fused form."""
    cd = registry.get(name)
    with cd.model(n) as g, cd.model(n) as f:
        for m, mode in ((g, MODE_GRAPH), (f, MODE_FUSED)):
            m.begin(SEED)
            m.run_cycles(9, mode)
        assert (g.hashes() == f.hashes()).all()
        for lane in sorted({0, n // 2, n - 1}):
            assert g.lane_state(lane) == f.lane_state(lane)


@pytest.mark.gpu
def test_packed_graph_done_lanes(gpu):
    """Done lanes inside a group of four keep every byte of their state; the
    lanes beside them go on."""
    cd = registry.get("net_tiny")
    n = 300
    done = np.zeros(n, np.uint8)
    done[[0, 5, 6, 7, 8, 9, 10, 11, 130, 255, 256, 299]] = 1
    with cd.model(n) as m, cd.model(n) as f:
        for x, mode in ((m, MODE_GRAPH), (f, MODE_FUSED)):
            x.begin(SEED)
            x.run_cycles(6, mode)
            before = [x.lane_state(k) for k in (5, 130, 299)]
            x.set_done(done)
            x.run_cycles(5, mode)
            assert [x.lane_state(k) for k in (5, 130, 299)] == before
            x.set_done(np.zeros(n, np.uint8))
            x.run_cycles(4, mode)
        assert (m.hashes() == f.hashes()).all()
        for k in (0, 1, 4, 5, 12, 130, 131, 254, 255, 257, 298, 299):
            assert m.lane_state(k) == f.lane_state(k)


@pytest.mark.gpu
def test_packed_graph_clock_differs_per_lane(gpu):
    """A rising clock in some lanes of a group of four only."""
    cd = registry.get("net_tiny")
    n, cycles = 22, 8
    up = np.array([(k * 7 + 3) % 3 != 0 for k in range(n)])
    ref = oracle.netlist_run(registry.table_bytes("net_tiny"), SEED, nstim=n, cycles=cycles)
    with cd.model(n) as m:
        h = np.full(n, 0xcbf29ce484222325, dtype=np.uint64)
        for c in range(cycles):
            # the lanes of `up` rise in the first half, the others in the second
            for half in (up, ~up):
                pi = np.array([oracle.stim(SEED, s, c, 0) & 0xffff for s in range(n)], np.uint16)
                m.set_port("pi", pi)
                m.set_port("clk", np.zeros(n, np.uint8))
                m.eval()
                m.set_port("clk", half.astype(np.uint8))
                m.eval()
                po = m.get_port("po")
                for s in np.nonzero(half)[0]:
                    h[s] = oracle.fnv(int(po[s]).to_bytes(2, "little"), int(h[s]))
    assert (h == ref).all()
