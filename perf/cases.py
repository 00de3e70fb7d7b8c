"""Performance cases: the work a user of the simulator has it do, each case
one pass through the public Python API (models, batched queues, input streams,
host-driven eval, the gate-net engine) from the design's reset state.

A case is a dict of plain values:

* ``kind`` "cycles": a model's state restored from a device checkpoint taken
  after set-up, ``begin``, ``run_cycles`` in one form, the per-stimulus hashes;
* ``kind`` "stream": the same with every input word read from a device buffer
  and every output word captured into another (both returned);
* ``kind`` "queue": a batched workload of uneven cycle budgets;
* ``kind`` "eval": a host-driven testbench: ports set, clk = 0 and clk = 1
  evaluated, the outputs read back, every clock;
* ``kind`` "gatenet": a netlist run as data by the gate-net engine.

Every output is a whole number, so the results have to be the same bits.
"""
import math

import numpy as np
import torch

from rtlflow_amd.designs import registry, rv32i
from rtlflow_amd.gatenet import GateNet
from rtlflow_amd.model import MODE_BITPLANE, MODE_FUSED, MODE_GRAPH

# Per design: packed state bytes a stimulus has to carry from cycle to cycle,
# and the operations of one stimulus-cycle: for the per-lane designs the
# front end's instruction count of two evals, for the netlists live gates
# over the 64 stimuli of a machine word.
DESIGNS = {
    "net_small": dict(state=24, ops=779 / 64.0),
    "net2": dict(state=238, ops=8138 / 64.0),
    "net_ram": dict(state=28, ops=778 / 64.0),
    "net5s": dict(state=660, ops=21080 / 64.0),
    "net5_small": dict(state=140, ops=2776 / 64.0),
    "net5": dict(state=6000, ops=178358 / 64.0),
    "alu": dict(state=156, ops=122.0),
    "systolic": dict(state=2051, ops=11234.0),
    "rv32i": dict(state=185, ops=1114.0),
}
MODES = {"graph": MODE_GRAPH, "fused": MODE_FUSED, "bitplane": MODE_BITPLANE}


def listed():
    return [
        # the smallest call: one 64-stimulus group of a small netlist for a
        # few cycles, as an interactive check or a unit test runs it
        dict(name="netlist_smallest", kind="cycles", design="net_small", lib="net_small", form="bitplane",
             stimuli=64, cycles=16, chunk=512, threads=512, lane_pad=0, multiwave=False),
        # an ordinary regression of a gate-level netlist, a ragged number of stimuli
        dict(name="netlist_ragged", kind="cycles", design="net2", lib="net2", form="bitplane",
             stimuli=5000, cycles=333, chunk=512, threads=512, lane_pad=0, multiwave=False),
        # the headline batch: 65,536 stimuli x 2,000 cycles of the 20,000-gate netlist
        dict(name="netlist_batch", kind="cycles", design="net2", lib="net2", form="bitplane",
             stimuli=65536, cycles=2000, chunk=2048, threads=512, lane_pad=0, multiwave=False),
        # user stimulus streamed from device memory, every output captured
        dict(name="netlist_stream", kind="stream", design="net2", lib="net2", form="bitplane",
             stimuli=20000, cycles=200, chunk=512, threads=512),
        # the plain form (one kernel per mtask, a graph per clock cycle),
        # which takes any design
        dict(name="netlist_graph", kind="cycles", design="net2", lib="net2", form="graph",
             stimuli=65536, cycles=16, chunk=512, threads=512, lane_pad=0, multiwave=False),
        # a small word-level design for many cycles
        dict(name="alu_long", kind="cycles", design="alu", lib="alu_tuned", form="fused",
             stimuli=1024, cycles=10000, chunk=512, threads=512, lane_pad=64, multiwave=False),
        # a wide word-level design (16 x 16 multiply-accumulates, 4,096-bit chain)
        dict(name="systolic", kind="cycles", design="systolic", lib="systolic_tuned", form="fused",
             stimuli=8192, cycles=1000, chunk=512, threads=512, lane_pad=0, multiwave=True),
        # processors running their own programs to uneven lengths
        dict(name="rv32i_queue", kind="queue", design="rv32i", lib="rv32i_tuned", form="fused",
             stimuli=2048, lanes=512, median=5000, lo=1000, hi=100000, threads=512),
        # a netlist with RAMs, uneven lengths
        dict(name="ram_netlist_queue", kind="queue", design="net5s", lib="net5s", form="bitplane",
             stimuli=4096, lanes=4096, median=500, lo=50, hi=5000, threads=1024),
        # a host-driven testbench: a few clocks, ports set and read each
        dict(name="alu_host_eval", kind="eval", design="alu", lib="alu", stimuli=300, cycles=8),
        # a small netlist as data, ragged
        dict(name="gatenet_small", kind="gatenet", design="net5_small", stimuli=200, median=200, lo=20, hi=2000),
        # half a million gates as data
        dict(name="gatenet_large", kind="gatenet", design="net5", stimuli=4096, median=500, lo=50, hi=5000),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread evenly over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    pick = rng.choice(["bitplane", "bitplane", "bitplane", "stream", "graph", "fused", "fused", "rv32i",
                       "ramqueue", "eval", "gatenet_small", "gatenet", "gatenet"])
    if pick == "bitplane":
        design = rng.choice(["net2", "net2", "net_small", "net_ram"])
        return dict(kind="cycles", design=design, lib=design, form="bitplane", stimuli=_log(rng, 17, 65536),
                    cycles=_log(rng, 3, 2000), chunk=rng.choice([512, 2048]), threads=rng.choice([256, 512, 512]),
                    lane_pad=0, multiwave=False)
    if pick == "stream":
        design = rng.choice(["net2", "net_small"])
        return dict(kind="stream", design=design, lib=design, form=rng.choice(["bitplane", "bitplane", "fused"])
                    if design == "net_small" else "bitplane", stimuli=_log(rng, 33, 20000),
                    cycles=_log(rng, 5, 256), chunk=512, threads=512)
    if pick == "graph":
        design = rng.choice(["net2", "net_small", "alu", "systolic"])
        return dict(kind="cycles", design=design, lib=design, form="graph",
                    stimuli=_log(rng, 65, 16384 if design == "systolic" else 65536), cycles=_log(rng, 2, 16),
                    chunk=512, threads=512, lane_pad=0, multiwave=False)
    if pick == "fused":
        design, lib, mw, most = rng.choice([("alu", "alu_tuned", False, 16384), ("alu", "alu", False, 16384),
                                            ("systolic", "systolic_tuned", True, 8192),
                                            ("net_small", "net_small", True, 16384),
                                            ("net_small", "net_small", False, 16384)])
        return dict(kind="cycles", design=design, lib=lib, form="fused", stimuli=_log(rng, 50, most),
                    cycles=_log(rng, 10, 2000), chunk=512, threads=512, lane_pad=0, multiwave=mw)
    if pick == "rv32i":
        n = _log(rng, 40, 1024)
        return dict(kind="queue", design="rv32i", lib=rng.choice(["rv32i_tuned", "rv32i"]), form="fused",
                    stimuli=n, lanes=max(1, n // rng.choice([1, 4])), median=_log(rng, 500, 5000), lo=100,
                    hi=50000, threads=512)
    if pick == "ramqueue":
        n = _log(rng, 64, 4096)
        return dict(kind="queue", design=rng.choice(["net5s", "net_ram"]), lib="", form="bitplane", stimuli=n,
                    lanes=max(1, n // rng.choice([1, 1, 2])), median=_log(rng, 50, 500), lo=10, hi=2500,
                    threads=rng.choice([512, 1024]))
    if pick == "eval":
        design = rng.choice(["alu", "net_small", "systolic"])
        return dict(kind="eval", design=design, lib=design, stimuli=_log(rng, 1, 4096), cycles=_log(rng, 2, 12))
    if pick == "gatenet_small":
        return dict(kind="gatenet", design="net5_small", stimuli=_log(rng, 1, 4096), median=_log(rng, 10, 200),
                    lo=5, hi=2000)
    return dict(kind="gatenet", design="net5", stimuli=_log(rng, 30, 4096), median=_log(rng, 20, 300), lo=10,
                hi=3000)


def _seed64(seed):
    return (seed * 0x9E3779B97F4A7C15 + 0x52544C46) & ((1 << 64) - 1)


def _lib(case):
    return registry.get(case.get("lib") or case["design"])


def _budgets(case, seed):
    return rv32i.budgets(seed, case["stimuli"], median=case["median"], lo=case["lo"], hi=case["hi"])


def _checkpoint(m):
    """A device-resident copy of the model's state."""
    m.sync()
    nb = m.checkpoint_bytes()
    ck = torch.empty(nb, dtype=torch.uint8, device="cuda")
    m.checkpoint_to(ck.data_ptr(), nb)
    m.sync()
    return ck


def prepare(case, seed):
    kind, n = case["kind"], case["stimuli"]
    s = {"case": case, "seed": _seed64(seed)}
    if kind == "gatenet":
        s["net"] = GateNet(registry.gatenet_program(case["design"]), n)
        s["budgets"] = _budgets(case, seed)
        return s
    cd = _lib(case)
    if kind == "queue":
        m = cd.model(case["lanes"], bitplane_threads=case["threads"])
        if case["design"] == "rv32i":
            m.set_mem_images("imem", rv32i.programs(s["seed"], np.arange(n)))
        s.update(model=m, budgets=_budgets(case, seed))
        return s
    if kind == "eval":
        m = cd.model(n)
        m.eval()
        rng = np.random.default_rng(seed)
        ports = [p for p in cd.manifest["ports"] if p["dir"] == 0 and p["name"] != "clk"]
        s["inputs"] = [{p["name"]: _port_values(rng, p, n) for p in ports} for _ in range(case["cycles"])]
        s["outputs"] = [p["name"] for p in cd.manifest["ports"] if p["dir"] == 1]
        s["low"], s["high"] = np.zeros(n, np.uint8), np.ones(n, np.uint8)
        s.update(model=m, ck=_checkpoint(m))
        return s
    mode = MODES[case["form"]]
    m = cd.model(n, fused_chunk=case["chunk"], bitplane_threads=case["threads"],
                 lane_pad=case.get("lane_pad", 0), fused_multiwave=int(case.get("multiwave", False)))
    m.begin(s["seed"])
    m.run_cycles(0, mode)
    s.update(model=m, mode=mode, ck=_checkpoint(m))
    if kind == "stream":
        nin, nout = m.stream_words()
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        s["x"] = torch.randint(-2**63, 2**63 - 1, (case["cycles"], nin, n), dtype=torch.int64, device="cuda",
                               generator=g)
        s["y"] = torch.zeros((case["cycles"], nout, n), dtype=torch.int64, device="cuda")
        m.set_input_stream(s["x"])
        m.set_output_capture(s["y"])
    return s


def _port_values(rng, p, n):
    """Uniform values of port ``p`` for n lanes, in its storage words."""
    dt = {0: np.uint8, 1: np.uint16, 2: np.uint32, 3: np.uint64}[p["cls"]]
    bits = np.dtype(dt).itemsize * 8
    out = np.empty((n, p["words"]), dt)
    for w in range(p["words"]):
        wide = min(bits, p["width"] - bits * w)
        out[:, w] = rng.integers(0, 2**wide - 1, n, dtype=np.uint64, endpoint=True).astype(dt)
    return out[:, 0] if p["words"] == 1 else out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "gatenet":
        return state["net"].run(GateNet.BITPLANE, state["seed"], state["budgets"])[0]
    m = state["model"]
    if kind == "queue":
        return m.submit_queue(state["seed"], state["budgets"], mode=MODES[case["form"]])
    ck = state["ck"]
    m.restore_from(ck.data_ptr(), ck.numel())
    if kind == "eval":
        out = []
        for values in state["inputs"]:
            for name, v in values.items():
                m.set_port(name, v)
            m.set_port("clk", state["low"])
            m.eval()
            m.set_port("clk", state["high"])
            m.eval()
            out += [m.get_port(name) for name in state["outputs"]]
        return out
    m.begin(state["seed"])
    m.run_cycles(case["cycles"], state["mode"])
    hashes = m.hashes()
    return [hashes, state["y"]] if kind == "stream" else hashes


def work(case):
    """What no implementation can do without: each stimulus's state read and
    written once, its streams and hash; the live logic of every stimulus-cycle."""
    d, n = DESIGNS[case["design"]], case["stimuli"]
    nbytes = n * (2 * d["state"] + 8)
    if "median" in case:
        # a lognormal of sigma 1 has a mean of 1.65 medians
        cycles = n * 1.65 * case["median"]
        nbytes += 4 * n + (n * 4 * rv32i.PROGRAM_WORDS if case["design"] == "rv32i" else 0)
    else:
        cycles = n * case["cycles"]
        if case["kind"] == "stream":
            nbytes += 16 * cycles
        elif case["kind"] == "eval":
            nbytes += 16 * cycles
    return {"bytes": float(nbytes), "flops": float(cycles * d["ops"])}


def tolerance(case):
    return "exact"


def exact(case, seed):
    return None   # hashes and port values are whole numbers: compared bit for bit
