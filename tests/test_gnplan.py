"""The LDS planner of the gate-net engine (csrc/rf_gnplan.h) on the CPU: a
model of the kernel (gnplan_host.cpp) runs the planned wavefront programs and
must hash as the C oracle does, over netlists with and without RAMs, ragged
levels and outputs or flip-flops driven by inputs, flip-flops or RAM data;
within a level no row may read what another writes."""
import ctypes as C
import resource
import subprocess
from pathlib import Path

import numpy as np
import pytest

import lds_nets
import oracle
from rtlflow_amd import gatenet as gn
from rtlflow_amd.designs.netlist import MUX, GateTable, generate

ROOT = Path(__file__).resolve().parent


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    so = tmp_path_factory.mktemp("gnplan") / "gnplan.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-Wl,-Bsymbolic", "-I",
                    str(ROOT.parent / "rtlflow_amd" / "csrc"),
                    str(ROOT / "gnplan_host.cpp"), "-o", str(so)], check=True)
    return C.CDLL(str(so))


def plan_run(host, prog, waves, seed, budgets, pb=1):
    b = np.asarray(budgets, np.uint32)
    out, info = np.zeros(len(b), np.uint64), np.zeros(7, np.uint32)
    rc = host.gnplan_run(prog.ctypes.data_as(C.c_void_p), waves, pb, C.c_uint64(seed), b.ctypes.data_as(C.c_void_p),
                         len(b), out.ctypes.data_as(C.c_void_p), info.ctypes.data_as(C.c_void_p))
    return rc, out, info


NETS = [dict(n_gates=900, n_ff=90, n_pi=100, n_po=40, depth=9, n_rams=2, ram_depth=48, ram_width=20),
        dict(n_gates=5000, n_ff=700, n_pi=64, n_po=64, depth=30),
        dict(n_gates=9000, n_ff=1500, n_pi=128, n_po=64, depth=8),
        dict(n_gates=40, n_ff=5, n_pi=3, n_po=2, depth=3),
        dict(n_gates=3000, n_ff=300, n_pi=128, n_po=7, depth=6, n_rams=3, ram_depth=64, ram_width=64)]


@pytest.mark.parametrize("k", range(len(NETS)))
@pytest.mark.parametrize("waves", [1, 16])
def test_planned_programs_hash_as_the_oracle(host, k, waves):
    table = generate(seed=0x51A + k, **NETS[k])[1]
    budgets = [7, 0, 1, 30]
    prog = gn.program(table, threads=None)
    rc, got, info = plan_run(host, prog, waves, 0xABCDEF, budgets)
    assert rc == 0
    want = oracle.netlist_run(table.to_bytes(), 0xABCDEF, len(budgets), budgets=budgets)
    assert (got == want).all()
    assert info[0] < table.first_gate + table.n_gates + 2 * table.n_pi


def test_sources_at_outputs_flip_flops_and_ports(host):
    """Outputs, D inputs and RAM ports that are inputs, flip-flops (a shift
    chain among them) or RAM data, several flip-flops on one value, outputs
    of equal gates."""
    table = generate(seed=0x77, n_gates=300, n_ff=40, n_pi=20, n_po=10, depth=5, n_rams=1, ram_depth=16,
                     ram_width=8)[1]
    g0 = table.first_gate
    ff = table.n_pi + np.arange(table.n_ff)
    table.ff_d[1:8] = ff[0:7]                       # a shift chain
    table.ff_d[8:12] = 3                            # an input, four times
    table.ff_d[12] = table.n_pi + table.n_ff + 2    # RAM data
    table.ff_d[13:17] = g0 + 17                     # one gate, four times
    table.po[0:4] = [0, ff[7], table.n_pi + table.n_ff, g0 + 17]
    table.ram_addr[0][:2] = [1, ff[3]]
    table.ram_wdata[0][:3] = [2, ff[12], table.n_pi + table.n_ff + 5]
    budgets = [25, 3, 40]
    for waves in (1, 4):
        rc, got, _ = plan_run(host, gn.program(table, threads=None), waves, 99, budgets)
        assert rc == 0
        assert (got == oracle.netlist_run(table.to_bytes(), 99, len(budgets), budgets=budgets)).all()


def test_programs_out_of_level_order_are_not_planned(host):
    """A cone that lacks a gate, or a record that reads its own level, keeps
    the level-by-level form."""
    table = generate(seed=5, n_gates=400, n_ff=30, n_pi=16, n_po=8, depth=6)[1]
    prog = gn.program(table, threads=None)
    n_cone, off = int(prog[14]), int(prog[22])
    assert plan_run(host, prog, 4, 1, [2])[0] == 0
    bad = prog.copy()
    bad[off + 4 * (n_cone - 1)] ^= 1 << 29          # another operator in the cone
    assert plan_run(host, bad, 4, 1, [2])[0] == 1
    full = int(prog[21])
    bad = prog.copy()
    bad[full + 1] = bad[full + 4] & ((1 << 29) - 1)  # the first record reads the second's node
    assert plan_run(host, bad, 4, 1, [2])[0] == 1


def test_deep_chain_plans_in_memory_linear_in_its_depth(host, monkeypatch):
    """20,000 levels of one multiplexer each: the plan's tables grow with the
    depth, not with its square (a key of level and death in 32 bits would wrap
    from 16,384 levels on)."""
    n, n_pi = 20000, 8
    rng = np.random.default_rng(9)
    first = n_pi + 1
    gin = np.zeros((n, 3), np.uint32)
    gin[:, 0] = rng.integers(0, n_pi, n)
    gin[:, 1] = np.arange(first - 1, first - 1 + n)     # the gate before (first: the flip-flop)
    gin[:, 2] = rng.integers(0, first, n)
    swap = rng.random(n) < 0.5
    gin[swap, 1], gin[swap, 2] = gin[swap, 2], gin[swap, 1].copy()
    table = GateTable(n_pi, 1, 0, np.full(n, MUX, np.uint8), gin, np.array([first + n // 2], np.uint32),
                      np.array([first + n - 1, first + n - 2], np.uint32))
    monkeypatch.setattr(gn, "gate_levels", lambda t: np.arange(1, n + 1, dtype=np.int32))
    budgets = [3, 1]
    before = resource.getrusage(resource.RUSAGE_SELF).ru_maxrss
    rc, got, info = plan_run(host, gn.program(table, threads=None), 16, 0x77, budgets)
    assert rc == 0 and info[2] == n + 1
    assert resource.getrusage(resource.RUSAGE_SELF).ru_maxrss - before < 1 << 20    # KiB
    assert (got == oracle.netlist_run(table.to_bytes(), 0x77, len(budgets), budgets=budgets)).all()


def test_plan_without_memory_is_no_plan(host):
    """Whichever allocation of the planner fails, the program is not planned
    (it runs level by level) and no exception leaves the planner."""
    prog = gn.program(generate(seed=0x51A, **NETS[0])[1], threads=None)
    used = C.c_long(0)

    def width(left, lds=160 * 1024):
        return host.gnplan_width(prog.ctypes.data_as(C.c_void_p), 16, C.c_uint64(lds), C.c_long(left), C.byref(used))

    assert width(-1) == 4
    total = used.value
    assert total > 100
    for left in sorted({0, 1, 2, *range(0, total, max(1, total // 97)), total - 1}):
        assert width(left) == 0, left
    assert width(total) == 4
    assert width(-1, lds=256) == 0


@pytest.mark.parametrize("pb", [2, 4])
@pytest.mark.parametrize("waves", [1, 16])
def test_wider_planes_hash_as_the_oracle(host, pb, waves):
    """Addresses and bank orders of 2- and 4-byte planes, batches of 4
    wavefront rows (one wavefront) and of 1."""
    batches = set()
    for k in range(len(NETS)):
        table = generate(seed=0x51A + k, **NETS[k])[1]
        budgets = [7, 0, 12]
        rc, got, info = plan_run(host, gn.program(table, threads=None), waves, 0xABCDEF, budgets, pb)
        assert rc == 0
        assert (got == oracle.netlist_run(table.to_bytes(), 0xABCDEF, len(budgets), budgets=budgets)).all()
        batches.add(int(info[5]))
    assert batches == ({1, 4} if waves == 1 else {1})


@pytest.mark.parametrize("name", lds_nets.NETS)
def test_instances_of_the_netlists_that_run_on_the_gpu(host, name):
    """The plane width and the batches that each netlist of the GPU test plans
    to, and its planned program against the oracle."""
    width, batch, kw, _ = lds_nets.NETS[name]
    table = lds_nets.table(name)
    prog = gn.program(table, threads=None)
    used = C.c_long(0)
    assert host.gnplan_width(prog.ctypes.data_as(C.c_void_p), 16, C.c_uint64(lds_nets.LDS_BYTES), C.c_long(-1),
                             C.byref(used)) == width
    rc, got, info = plan_run(host, prog, 16, 5, [3, 1], width)
    assert rc == 0 and info[5] == batch
    assert info[6] > 14 or name != "20 RAMs"
    assert (got == oracle.netlist_run(table.to_bytes(), 5, 2, budgets=[3, 1])).all()
