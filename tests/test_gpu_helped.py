"""GPU: the fused kernel with helper wavefronts (inputs a stage of eight cycles
ahead, hash a stage behind) against the graph form, where a stage or a group of
64 lanes is cut. Whole numbers: exact."""
import numpy as np
import pytest

from rtlflow_amd.designs import registry
from rtlflow_amd.model import MODE_FUSED, MODE_GRAPH


def _same(f, g, n):
    assert (f.hashes() == g.hashes()).all()
    for lane in sorted({0, n // 2, n - 1}):
        assert f.lane_state(lane) == g.lane_state(lane), lane


@pytest.mark.gpu
@pytest.mark.parametrize("n,runs", [(1, (1,)), (63, (7, 8)), (64, (9,)), (65, (16, 1, 17)), (300, (15, 25))])
def test_helped_matches_graph(gpu, n, runs):
    cd = registry.get("alu")
    with cd.model(n) as f, cd.model(n) as g:
        for m, mode in ((f, MODE_FUSED), (g, MODE_GRAPH)):
            m.begin(0xA1, stim0=3)
            for c in runs:
                m.run_cycles(c, mode)
        _same(f, g, n)


@pytest.mark.gpu
def test_helped_done_lanes_and_chunks(gpu):
    """A whole group done, single lanes done, and launches of five cycles."""
    cd = registry.get("alu")
    n = 200
    done = np.zeros(n, np.uint8)
    done[64:128] = 1
    done[[0, 5, 63, 129, 199]] = 1
    with cd.model(n, fused_chunk=5) as f, cd.model(n) as g:
        for m, mode in ((f, MODE_FUSED), (g, MODE_GRAPH)):
            m.begin(0xA2)
            m.run_cycles(11, mode)
            before = [m.lane_state(k) for k in (0, 70, 199)]
            m.set_done(done)
            m.run_cycles(12, mode)
            assert [m.lane_state(k) for k in (0, 70, 199)] == before
            m.set_done(np.zeros(n, np.uint8))
            m.run_cycles(9, mode)
        _same(f, g, n)
        for lane in (5, 64, 100, 129, 130):
            assert f.lane_state(lane) == g.lane_state(lane), lane


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["gated", "kat_shift"])
def test_helped_other_designs(gpu, name):
    """A derived clock (three helpers) and wide operands (two): cut stages,
    done lanes, launches of five cycles."""
    cd = registry.get(name)
    n = 130
    done = np.zeros(n, np.uint8)
    done[[0, 63, 64, 100, 129]] = 1
    with cd.model(n, fused_chunk=5) as f, cd.model(n) as g:
        for m, mode in ((f, MODE_FUSED), (g, MODE_GRAPH)):
            m.begin(0xA3)
            m.run_cycles(9, mode)
            m.set_done(done)
            m.run_cycles(17, mode)
        _same(f, g, n)
