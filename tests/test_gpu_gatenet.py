"""GPU parity of the gate-net engine (include/rf_gatenet.h) against the C
oracle: a small netlist of configuration 5's shape in both forms with ragged
lane counts and uneven budgets, and configuration 5 at its stated size
(500,000 gates, 50,000 flip-flops, eight 1,024 x 64-bit RAMs, 128 inputs,
4,096 stimuli with lognormal budgets) on a sample of stimuli, with the
heuristic and the learned partitions."""
import numpy as np
import pytest

import lds_nets
import oracle
from rtlflow_amd.designs import registry, rv32i
from rtlflow_amd.gatenet import GateNet, program

SEED = registry.SEED_CFG[5]


@pytest.mark.gpu
@pytest.mark.parametrize("lanes", [130, 1024])
@pytest.mark.parametrize("mode", [GateNet.GRAPH, GateNet.BITPLANE])
def test_gatenet_small_matches_oracle(gpu, lanes, mode):
    tb = registry.gatenet_table("net5_small")
    prog = registry.gatenet_program("net5_small")
    rng = np.random.default_rng(lanes + mode)
    budgets = rng.integers(0, 40, size=lanes).astype(np.uint32)
    print(f"gatenet net5_small lanes={lanes} mode={mode}", flush=True)
    with GateNet(prog, lanes) as g:
        got, _ = g.run(mode, SEED, budgets)
    want = oracle.netlist_run(tb, SEED, lanes, budgets=budgets)
    assert (got == want).all(), f"{int((got != want).sum())} of {lanes} differ"


def _net5_budgets(n, median):
    return rv32i.budgets(SEED, n, median=median, lo=1, hi=3 * median)


@pytest.mark.gpu
def test_config5_full_size_bitplane_matches_oracle(gpu):
    """4,096 stimuli, lognormal budgets (median 24): the first and last 16
    stimuli against the oracle."""
    n = 4096
    tb = registry.gatenet_table("net5")
    prog = registry.gatenet_program("net5")
    budgets = _net5_budgets(n, 24)
    print(f"gatenet net5 bitplane lanes={n} max budget={int(budgets.max())}", flush=True)
    with GateNet(prog, n) as g:
        got, ms = g.run(GateNet.BITPLANE, SEED, budgets)
    for s0 in (0, n - 16):
        want = oracle.netlist_run(tb, SEED, 16, stim0=s0, budgets=budgets[s0:s0 + 16])
        assert (got[s0:s0 + 16] == want).all(), s0


@pytest.mark.gpu
@pytest.mark.parametrize("name,lanes,warm", [("net5", 200, 1000), ("net5_small", 1, 0), ("net5_small", 33, 12),
                                             ("net5_small", 9000, 20)])
def test_lds_form_matches_oracle(gpu, name, lanes, warm):
    """After ``warm`` cycles the handle runs in LDS: ragged last workgroups,
    budgets of 0, the same handle twice, and hashes equal to the level-by-level
    form's (the first, short runs)."""
    tb = registry.gatenet_table(name)
    budgets = np.random.default_rng(lanes).integers(0, 40, size=lanes).astype(np.uint32)
    budgets[0] = 40
    print(f"gatenet lds {name} lanes={lanes}", flush=True)
    with GateNet(registry.gatenet_program(name), lanes) as g:
        first, _ = g.run(GateNet.BITPLANE, SEED, np.minimum(budgets, 2))
        g.run(GateNet.BITPLANE, SEED, np.full(lanes, warm, np.uint32))
        got, _ = g.run(GateNet.BITPLANE, SEED, budgets)
        assert g.nodes_per_cycle(GateNet.BITPLANE) == 0
        again, _ = g.run(GateNet.BITPLANE, SEED, np.minimum(budgets, 2))
    assert (first == again).all()
    k = min(lanes, 16 if name == "net5" else 512)
    for s0 in {0, lanes - k}:
        want = oracle.netlist_run(tb, SEED, k, stim0=s0, budgets=budgets[s0:s0 + k])
        assert (got[s0:s0 + k] == want).all(), s0


@pytest.mark.gpu
@pytest.mark.parametrize("name", lds_nets.NETS)
def test_lds_instances_match_oracle(gpu, name):
    """Every instance of the LDS kernel, and more RAMs than wavefronts for
    them, against the oracle; a budget of 0 and a ragged last workgroup."""
    table = lds_nets.table(name)
    prog = program(table, threads=None)
    lanes = 41
    budgets = np.random.default_rng(7).integers(1, 30, size=lanes).astype(np.uint32)
    budgets[[3, 40]] = 0
    print(f"gatenet lds instance {name}", flush=True)
    with GateNet(prog, lanes) as g:
        # enough cycles that the handle plans (four launches a cycle at least)
        g.run(GateNet.BITPLANE, SEED, np.full(lanes, len(table.gate_type) // 64 + 1, np.uint32))
        assert g.nodes_per_cycle(GateNet.BITPLANE) == 0
        got, _ = g.run(GateNet.BITPLANE, SEED, budgets)
    want = oracle.netlist_run(table.to_bytes(), SEED, lanes, budgets=budgets)
    assert (got == want).all(), f"{int((got != want).sum())} of {lanes} differ"


@pytest.mark.gpu
def test_lds_form_begins_where_planning_pays(gpu):
    """net5_small (6,000 gates, 24 launches a cycle) pays for its plan from 16
    cycles on, the coming run's included."""
    prog = registry.gatenet_program("net5_small")
    print("gatenet lds net5_small planning", flush=True)
    with GateNet(prog, 40) as g:
        for cycles, planned in ((10, False), (5, False), (1, True), (3, True)):
            g.run(GateNet.BITPLANE, SEED, np.full(40, cycles, np.uint32))
            assert (g.nodes_per_cycle(GateNet.BITPLANE) == 0) == planned, cycles


@pytest.mark.gpu
def test_lds_form_across_launches(gpu):
    """A budget past one launch's 16,384 cycles: the state goes on in the next
    launch (a lane next to it stops before, another just at the boundary)."""
    budgets = np.array([16390, 16383, 16384, 20, 0], np.uint32)
    tb = registry.gatenet_table("net5_small")
    print("gatenet lds net5_small two launches", flush=True)
    with GateNet(registry.gatenet_program("net5_small"), len(budgets)) as g:
        got, _ = g.run(GateNet.BITPLANE, SEED, budgets)
    assert (got == oracle.netlist_run(tb, SEED, len(budgets), budgets=budgets)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("schedule", ["heuristic", "learned"])
def test_config5_full_size_graph_form_matches_oracle(gpu, schedule):
    if schedule not in registry.gatenet_meta("net5")["schedules"]:
        pytest.skip("no learned partition chosen for net5")
    n = 4096
    tb = registry.gatenet_table("net5")
    prog = registry.gatenet_program("net5", schedule)
    budgets = _net5_budgets(n, 4)
    print(f"gatenet net5 graph {schedule} lanes={n} max budget={int(budgets.max())}", flush=True)
    with GateNet(prog, n) as g:
        got, ms = g.run(GateNet.GRAPH, SEED, budgets)
    for s0 in (0, n - 16):
        want = oracle.netlist_run(tb, SEED, 16, stim0=s0, budgets=budgets[s0:s0 + 16])
        assert (got[s0:s0 + 16] == want).all(), s0
