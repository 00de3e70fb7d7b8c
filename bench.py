"""Throughput benchmark: stimulus-cycles/s on one MI355X.

Workload: the seeded random gate-level netlist (20,000 gates, 2,000 flip-flops,
64 primary inputs, 64 primary outputs, depth 40), 65,536 stimuli x 2,000
cycles, 64-bit uniform inputs per cycle generated on the device, per-cycle
FNV-1a-64 output hash per stimulus.

A step is the whole workload from its start: the post-set-up model state is
restored from a device-resident checkpoint, the stimuli restart at cycle 0
(a fresh rf_begin) and all 2,000 cycles run in the bit-plane form (the
design lowered to single-bit logic, 64 stimuli per 64-bit word, node values
in LDS, one kernel launch). ``--steps`` steps are timed; every step
recomputes the same hashes, and the last step's are checked against the CPU
oracle on stimuli sampled from the first, middle and last workgroups and the
two sides of the workgroup-slot boundary.

Beside it, each measured once on a bounded number of cycles that does not
depend on ``--steps``: the fused per-lane kernel, the plain per-mtask hipGraph
form, the learned-vs-heuristic partition in the graph form, and the
bit-plane launch with its input words streamed from HBM (then with the
outputs captured too), checked against the generator run. The CPU
oracle is timed on a bounded sample as the reported CPU baseline. Optional
legs are skipped once ``--budget-s`` seconds have passed.
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time
from pathlib import Path

import numpy as np

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))
sys.path.insert(0, str(ROOT / "oracle"))

HBM_PEAK_GBS = 8000.0
CUS = 256
CLOCK_HZ = 2.4e9                     # MI355X peak engine clock
VALU_PEAK = CUS * 4 * 16 * CLOCK_HZ  # int32 lane-ops/s: 256 CUs x 4 SIMD x 16 lanes
WAVE64 = 64


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def cpu_threads() -> int:
    return max(1, min(16, os.cpu_count() or 1))


def run_form(cd, lanes, mode, cycles, seed, chunk, bp_threads=0):
    """One bounded run of ``cycles`` cycles from a fresh model; the model's
    set-up (initial blocks, time-0 settle) runs before the timed region."""
    with cd.model(lanes, fused_chunk=chunk, bitplane_threads=bp_threads) as m:
        m.begin(seed)
        m.run_cycles(0, mode)
        m.sync()
        m.reset_stats()
        t0 = time.perf_counter()
        m.run_cycles(cycles, mode)
        m.sync()
        dt = time.perf_counter() - t0
        st = m.stats()
        h = m.hashes()
    return dt, st, h


def sample_groups(lanes: int, slots: int):
    """64-lane groups to check: the first, the last of the first round of
    workgroup slots and the first of the second, the middle and the last."""
    ng = (lanes + 63) // 64
    gs = {0, ng // 2, ng - 1}
    if slots < ng:
        gs |= {slots - 1, slots}
    return sorted(g for g in gs if 0 <= g < ng)


def check_sample(table, seed, h, lanes, cycles, groups, per_group=64):
    """Compare the hashes of the sampled groups with the oracle."""
    import oracle
    bad = 0
    n = 0
    for g in groups:
        s0 = g * 64
        k = min(per_group, lanes - s0)
        ref = oracle.netlist_run(table, seed, nstim=k, cycles=cycles, stim0=s0, threads=cpu_threads())
        bad += int((h[s0:s0 + k] != ref).sum())
        n += k
    return bad == 0, n, bad


def profile_json(name: str):
    p = ROOT / "profiles" / name
    return json.loads(p.read_text()) if p.exists() else None


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--cycles", type=int, default=2000, help="cycles per stimulus in one step")
    ap.add_argument("--lanes", type=int, default=65536)
    ap.add_argument("--design", default="net2")
    ap.add_argument("--bp-chunk", type=int, default=2048,
                    help="cycles per bit-plane launch (the state stays in LDS across them)")
    ap.add_argument("--bp-threads", type=int, default=0,
                    help="bit-plane form: threads per 64-lane workgroup (0: the autotuned choice)")
    ap.add_argument("--chunk", type=int, default=512, help="cycles per fused launch")
    ap.add_argument("--fused-cycles", type=int, default=256,
                    help="cycles of the fused-form comparison (0: skip)")
    ap.add_argument("--graph-cycles", type=int, default=64,
                    help="cycles of the plain graph-form comparison (0: skip)")
    ap.add_argument("--stream-cycles", type=int, default=256,
                    help="cycles of the input-stream leg (0: skip)")
    ap.add_argument("--learned-cycles", type=int, default=64,
                    help="cycles of the learned-vs-heuristic partition comparison (0: skip)")
    ap.add_argument("--workload", default="netlist",
                    choices=["netlist", "alu", "systolic", "rv32i", "net5s", "net5"],
                    help="netlist (default, the headline) or one of the other synthetic designs")
    ap.add_argument("--check", type=int, default=64, help="stimuli checked per sampled group")
    ap.add_argument("--cpu-sample", type=int, default=0,
                    help="stimuli in the CPU baseline sample of the other workloads (0: the "
                         "workload's default, sized to a few seconds of CPU work)")
    ap.add_argument("--cpu-sample-netlist", type=int, default=1024,
                    help="stimuli in the netlist CPU baseline sample (x the full cycles)")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--budget-cap", type=int, default=0,
                    help="net5: cap every stimulus's budget (0: none; for short counter profiles)")
    ap.add_argument("--main-only", action="store_true",
                    help="run only the reported form: the headline's bit-plane steps, or another "
                         "workload's main leg (for counter profiles)")
    ap.add_argument("--budget-s", type=float, default=300.0,
                    help="optional legs (other forms, learned partition, CPU baseline) are "
                         "skipped once this many seconds have passed")
    ap.add_argument("--calibrate-copy", type=int, default=0, metavar="MB",
                    help="only run a plain device-to-device copy of MB megabytes three times "
                         "(the reference kernel for scaling rocprofv3 FETCH_SIZE / WRITE_SIZE)")
    args = ap.parse_args()
    if args.calibrate_copy:
        import torch
        n = args.calibrate_copy << 20
        src = torch.ones(n, dtype=torch.uint8, device="cuda")
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        print(json.dumps({"calibrate_copy_bytes": n, "launches": 3}), flush=True)
        return
    if args.gpus != 1:
        print(f"bench.py: this build runs on one GPU only (asked for {args.gpus}); "
              "stimuli shard trivially across GPUs but no multi-GPU path is built", file=sys.stderr)
        sys.exit(2)

    import torch
    if not torch.cuda.is_available():
        print("bench.py needs a GPU", file=sys.stderr)
        sys.exit(1)
    if args.workload != "netlist":
        return bench_other(args)
    return bench_netlist(args, torch)


def bench_netlist(args, torch):
    from rtlflow_amd.designs import registry
    from rtlflow_amd.model import MODE_BITPLANE, MODE_FUSED, MODE_GRAPH
    import oracle

    t_start = time.perf_counter()

    def budget_left(leg):
        if time.perf_counter() - t_start > args.budget_s:
            log(f"[bench] {leg}: skipped (past the {args.budget_s:.0f} s budget)")
            return False
        return True

    if args.main_only:
        # only the bit-plane steps (and their oracle sample)
        args.fused_cycles = args.graph_cycles = args.learned_cycles = args.stream_cycles = 0
        args.no_cpu = True
    seed = registry.SEED_CFG[2]
    cd = registry.get(args.design)
    man = cd.manifest
    table = registry.table_bytes(args.design)
    if not args.bp_threads:
        from rtlflow_amd.autotune import choice
        tuned = choice(args.design)
        args.bp_threads = (tuned["knobs"]["bp_threads"]
                           if tuned and tuned.get("form") == "bitplane" else 512)
    if not man.get("bitplane", {}).get("supported"):
        raise SystemExit(f"{args.design} has no bit-plane program: {man.get('bitplane')}")
    lanes, cycles, K, W = args.lanes, args.cycles, args.steps, args.warmup
    stim_cycles = lanes * cycles
    nt = args.bp_threads
    # workgroup slots of the bit-plane kernel: LDS per group decides how many
    # groups share a CU
    lds_per_group = man["bitplane"]["slots"] * 8
    per_cu = max(1, min(160 * 1024 // max(1, lds_per_group), 2048 // nt))
    slots = CUS * per_cu

    # ---- set-up (untimed): model, initial blocks + time-0 settle, and a
    # device-resident checkpoint of that state
    log(f"[bench] {args.design} bit-plane: {lanes} stimuli x {cycles} cycles per step, "
        f"{nt} threads per 64-lane group, {K} steps after {W} warm-up")
    m = cd.model(lanes, fused_chunk=args.bp_chunk, bitplane_threads=nt)
    m.begin(seed)
    m.run_cycles(0, MODE_BITPLANE)
    m.sync()
    nb = m.checkpoint_bytes()
    ck = torch.empty(nb, dtype=torch.uint8, device="cuda")
    m.checkpoint_to(ck.data_ptr(), nb)

    def step():
        m.restore_from(ck.data_ptr(), nb)
        m.begin(seed)
        m.run_cycles(cycles, MODE_BITPLANE)

    for _ in range(W):
        step()
    m.sync()
    m.reset_stats()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(K):
        step()
    m.sync()
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    st = m.stats()
    h = m.hashes()
    m.close()
    groups = sample_groups(lanes, slots)
    ok, nchk, bad = check_sample(table, seed, h, lanes, cycles, groups, args.check)
    value = K * stim_cycles / dt
    log(f"[bench] bitplane {dt:.3f}s for {K} steps, {value:.4g} stim-cycles/s; oracle sample of "
        f"{nchk} stimuli in groups {groups}: {'bit-exact' if ok else f'{bad} differ'}")
    forms = {"bitplane": {"seconds": dt, "steps": K, "value": value, "bit_exact_sample": ok,
                          "checked_stimuli": nchk, "checked_groups": groups, "cycles": cycles}}

    # ---- the other forms, once each on a bounded number of cycles
    for form, mode, cyc in (("fused", MODE_FUSED, args.fused_cycles),
                            ("graph", MODE_GRAPH, args.graph_cycles)):
        if not cyc or not budget_left(form):
            continue
        log(f"[bench] {args.design} form={form} lanes={lanes} cycles={cyc}")
        fdt, _, fh = run_form(cd, lanes, mode, cyc, seed, args.chunk)
        fok, fn, _ = check_sample(table, seed, fh, lanes, cyc, [0, (lanes + 63) // 64 - 1], args.check)
        forms[form] = {"seconds": fdt, "value": lanes * cyc / fdt, "bit_exact_sample": fok,
                       "checked_stimuli": fn, "cycles": cyc}
        log(f"[bench] form={form} {fdt:.3f}s {lanes * cyc / fdt:.4g} stim-cycles/s oracle_match={fok}")

    # ---- user input stream: the same launch shape with every input word
    # read from HBM instead of the generator, then with the outputs captured
    # as well; the stream holds the generator's own words, so the hashes must
    # equal the generator run's for every stimulus
    stream = None
    if args.stream_cycles and budget_left("input stream"):
        stream = bench_stream(args, torch, cd, man, lanes, nt, seed)

    # ---- learned partition: the plain graph form partitioned by the cost
    # model's choice of granularity against the instruction-count heuristic
    learned = None
    lname = args.design + "_learned"
    if args.learned_cycles and lname in registry.load_index() and budget_left("learned partition"):
        lcd = registry.get(lname)
        lc = args.learned_cycles
        res = {}
        for tag, c in (("heuristic", cd), ("learned", lcd)):
            log(f"[bench] partition={tag} graph form, {lanes} x {lc} cycles, "
                f"{c.manifest['mtasks']} mtasks")
            ldt, _, lh = run_form(c, lanes, MODE_GRAPH, lc, seed, args.chunk)
            res[tag] = (lanes * lc / ldt, lh, c.manifest["mtasks"])
        same = bool((res["heuristic"][1] == res["learned"][1]).all())
        lok, _, _ = check_sample(table, seed, res["learned"][1], lanes, lc, [0], 16)
        exact = same and lok
        sp = res["learned"][0] / res["heuristic"][0]
        learned = {"form": "graph", "cycles": lc,
                   "heuristic": res["heuristic"][0], "learned": res["learned"][0],
                   "heuristic_mtasks": res["heuristic"][2], "learned_mtasks": res["learned"][2],
                   "speedup": sp, "bit_exact": exact, "kept": bool(exact and sp > 1.0)}
        log(f"[bench] learned/heuristic graph throughput {sp:.3f} (bit-exact {exact})")

    # ---- roofline of the bit-plane kernel: algorithmic bytes per
    # stimulus-cycle are the bit-packed state read and written once
    state_bits = man["bitplane"]["state_bits"]
    b_alg = 2 * ((state_bits + 7) // 8)
    # (groups beyond the workgroup slots rotate through several launches of
    # one full round each: a launch's stimulus-cycles are the timed steps'
    # total over the launches)
    launches = max(1, st["bitplane_launches"])
    per_launch_ms = st["bitplane_ms"] / launches
    cyc_per_launch = min(cycles, args.bp_chunk)
    bytes_per_launch = b_alg * K * stim_cycles / launches
    achieved = bytes_per_launch / (per_launch_ms * 1e-3) / 1e9
    shape = {"lanes": lanes, "cycles_per_launch": cyc_per_launch, "bitplane_threads": nt,
             "launches_per_step": launches // K}
    traffic = None
    t = profile_json(f"{args.design}_bitplane_traffic.json")
    if t and all(t.get(k) == v for k, v in shape.items()):
        traffic = t["read_bytes"] + t["write_bytes"]
    # measured limits of the same launch shape from the committed SQ counters:
    # VALU issue (wave instructions over one per CU per clock), LDS bank
    # conflict cycles per CU-cycle, HBM traffic over peak bandwidth
    limits = sq_limits(f"{args.design}_bitplane_sq.json", shape, traffic)
    gates_m = man["bitplane"]["gates"][1]

    cpu = None
    if not args.no_cpu and budget_left("CPU baseline"):
        ns = args.cpu_sample_netlist
        th = cpu_threads()
        t0 = time.perf_counter()
        oracle.netlist_run(table, seed, nstim=ns, cycles=cycles, threads=th)
        cdt = time.perf_counter() - t0
        cpu = {"value": ns * cycles / cdt, "unit": "stimulus-cycles/s", "cores": th,
               "kind": "port", "nproc": os.cpu_count(),
               "sample": f"{ns} stimuli x {cycles} cycles of the same netlist and protocol "
                         f"({cdt:.1f} s), C oracle, one stimulus per thread on {th} threads"}

    line = {
        "metric": "stimulus-cycles/sec, bit-exact vs Verilator CPU; batched+learned vs plain GPU",
        "value": value,
        "unit": "stimulus-cycles/s",
        "n_gpus": 1,
        "steps": K,
        "warmup": W,
        "ms_per_step": dt / K * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "u64",
        "data": "synthetic (seeded netlist, on-device SplitMix64 stimulus)",
        "config": {"workload": f"random netlist 20k gates / 2k flops / 64 PI / 64 PO / depth 40, "
                               f"{lanes} stimuli x {cycles} cycles",
                   "design": args.design, "stimuli": lanes, "cycles": cycles,
                   "cycles_per_launch": cyc_per_launch, "launches_per_step": launches // K,
                   "form": "bitplane",
                   "bitplane_threads": nt, "mtasks": man["mtasks"]},
        "forms": forms,
        "learned_partition": learned,
        "input_stream": stream,
        "bit_exact_sample": all(v["bit_exact_sample"] for v in forms.values()),
        "roofline": {"bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": achieved / HBM_PEAK_GBS, "traffic": traffic,
                     "kernel": f"rf_bp_kernel<{nt}>", "alg_bytes_per_stimulus_cycle": b_alg,
                     "avg_launch_ms": per_launch_ms, "launches": launches, "limits": limits},
        "valu": {"gate_records_per_cycle": gates_m,
                 "note": "VALU issue of the bit-plane kernel is roofline.limits.valu_issue "
                         "(SQ_INSTS_VALU of the same launch shape)"},
        "cpu_baseline": cpu,
    }
    print(json.dumps(line), flush=True)


def generator_words_dev(torch, man, seed, nstim, c, device="cuda"):
    """The generator's input words of cycle ``c`` for stimuli [0, nstim) as
    an int64 [words, nstim] device tensor: SplitMix64 of seed ^ s * golden ^
    c << 8 ^ key (int64 arithmetic wraps like uint64; right shifts are made
    logical by masking)."""
    def lsr(z, k):
        return (z >> k) & ((1 << (64 - k)) - 1)

    def i64(v):
        v &= (1 << 64) - 1
        return v - (1 << 64) if v >= 1 << 63 else v

    gold = i64(0x9E3779B97F4A7C15)
    keys = [(p["stim_index"] << 3) | j for p in man["ports"] if p["dir"] == 0
            for j in range((p["width"] + 63) // 64)]
    s = torch.arange(nstim, dtype=torch.int64, device=device) * gold
    k = torch.tensor([i64(seed ^ (c << 8) ^ key) for key in keys], dtype=torch.int64, device=device)
    z = (s[None, :] ^ k[:, None]) + gold
    z = (z ^ lsr(z, 30)) * i64(0xBF58476D1CE4E5B9)
    z = (z ^ lsr(z, 27)) * i64(0x94D049BB133111EB)
    return z ^ lsr(z, 31)


def bench_stream(args, torch, cd, man, lanes, nt, seed):
    from rtlflow_amd.model import MODE_BITPLANE
    sc, reps = args.stream_cycles, 3
    nin, nout = man["streams"]["in_words"], man["streams"]["out_words"]
    xin = torch.empty((sc, nin, lanes), dtype=torch.int64, device="cuda")
    for c in range(sc):
        xin[c] = generator_words_dev(torch, man, seed, lanes, c)
    cap = torch.zeros((sc, nout, lanes), dtype=torch.int64, device="cuda")
    out = {"cycles": sc, "in_words": nin, "out_words": nout}
    with cd.model(lanes, fused_chunk=args.bp_chunk, bitplane_threads=nt) as m:
        # every run starts from the set-up state (device checkpoint)
        m.begin(seed)
        m.run_cycles(0, MODE_BITPLANE)
        m.sync()
        nb = m.checkpoint_bytes()
        ck = torch.empty(nb, dtype=torch.uint8, device="cuda")
        m.checkpoint_to(ck.data_ptr(), nb)
        m.run_cycles(sc, MODE_BITPLANE)
        ref = m.hashes()
        for tag, use_in, use_cap in (("generator", False, False), ("stream", True, False),
                                     ("stream_capture", True, True)):
            m.set_input_stream(xin if use_in else None)
            m.set_output_capture(cap if use_cap else None)
            m.sync()
            m.reset_stats()
            t0 = time.perf_counter()
            for _ in range(reps):
                m.restore_from(ck.data_ptr(), nb)
                m.begin(0 if use_in else seed)
                m.run_cycles(sc, MODE_BITPLANE)
            m.sync()
            dt = time.perf_counter() - t0
            st = m.stats()
            same = bool((m.hashes() == ref).all())
            per_ms = st["bitplane_ms"] / max(1, st["bitplane_launches"])
            kern_s = st["bitplane_ms"] * 1e-3          # every launch of the timed runs
            b = 2 * ((man["bitplane"]["state_bits"] + 7) // 8) + (8 * nin if use_in else 0) + \
                (8 * nout if use_cap else 0)
            out[tag] = {"value": reps * lanes * sc / dt, "kernel_value": reps * lanes * sc / kern_s,
                        "avg_launch_ms": per_ms, "launches": st["bitplane_launches"],
                        "alg_bytes_per_stimulus_cycle": b,
                        "hbm_frac": b * reps * lanes * sc / kern_s / (HBM_PEAK_GBS * 1e9),
                        "hashes_equal_generator_run": same}
            log(f"[bench] bitplane {tag}: {out[tag]['value']:.4g} stim-cycles/s "
                f"(kernel {out[tag]['kernel_value']:.4g}, {per_ms:.2f} ms per launch), "
                f"hashes equal the generator run: {same}")
        m.set_input_stream(None)
        m.set_output_capture(None)
    for tag in ("stream", "stream_capture"):
        out[tag]["kernel_vs_generator"] = out[tag]["kernel_value"] / out["generator"]["kernel_value"]
    del xin, cap
    torch.cuda.empty_cache()
    return out


# memory bytes a stimulus-cycle touches by design (T_mem): ALU two register
# reads and one write of 4 B; RV32I a 4 B fetch, at most 4 B of data and the
# register file's two reads and one write; systolic none
T_MEM = {"alu": 12, "systolic": 0, "rv32i": 20}


def sq_limits(sq_json, shape, traffic):
    """Measured limits of a launch shape from its committed SQ counters (one
    dispatch): VALU and LDS instruction issue (wave instructions over one per
    CU per clock), LDS bank-conflict cycles per CU-cycle, HBM traffic over
    peak bandwidth; None when no profile of that shape is committed."""
    q = profile_json(sq_json)
    if not (q and all(q.get(k) == v for k, v in shape.items())):
        return None
    ks = q["kernel_ns"] * 1e-9
    cu_cycles = CUS * CLOCK_HZ * ks
    limits = {"valu_issue": q["SQ_INSTS_VALU"] / cu_cycles,
              "lds_instr_issue": q["SQ_INSTS_LDS"] / cu_cycles,
              "lds_bank_conflict": q["SQ_LDS_BANK_CONFLICT"] / cu_cycles,
              "hbm_traffic": (traffic / ks / (HBM_PEAK_GBS * 1e9)) if traffic else None,
              "source": f"profiles/{sq_json}", "kernel_ns": q["kernel_ns"]}
    cand = {k: limits[k] for k in ("valu_issue", "lds_instr_issue", "lds_bank_conflict", "hbm_traffic")
            if isinstance(limits[k], float)}
    limits["highest"] = max(cand, key=cand.get)
    return limits


def roofline_line(b_alg, stim_cycles_per_launch, per_launch_ms, kernel, traffic_json=None, shape=None,
                  sq_json=None):
    achieved = b_alg * stim_cycles_per_launch / (per_launch_ms * 1e-3) / 1e9
    traffic = None
    t = profile_json(traffic_json) if traffic_json else None
    if t and shape and all(t.get(k) == v for k, v in shape.items()):
        traffic = t["read_bytes"] + t["write_bytes"]
    out = {"bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
           "frac": achieved / HBM_PEAK_GBS, "traffic": traffic, "kernel": kernel,
           "alg_bytes_per_stimulus_cycle": b_alg, "avg_launch_ms": per_launch_ms}
    if shape:
        out["shape"] = shape
    if sq_json and shape:
        out["limits"] = sq_limits(sq_json, shape, traffic)
    return out


def bench_other(args):
    """The other synthetic designs at their own sizes: ALU 1,024 x 10,000,
    systolic 8,192 x 5,000 (fused, tuned and graph forms), RV32I 16,384
    stimuli with lognormal budgets through the batched queue, beside the
    graph form at the median budget. A step is the whole workload."""
    from rtlflow_amd.designs import registry, rv32i
    from rtlflow_amd.model import MODE_FUSED, MODE_GRAPH
    import oracle
    wl = args.workload
    if wl == "net5s":
        return bench_net5s(args)
    if wl == "net5":
        return bench_net5(args)
    cfg = {"alu": 1, "rv32i": 3, "systolic": 4}[wl]
    seed = registry.SEED_CFG[cfg]
    cd = registry.get(wl)
    man = cd.manifest
    b_alg = 2 * man["bytes_seq"] + T_MEM[wl]
    th = cpu_threads()
    forms = {}
    if wl in ("alu", "systolic"):
        lanes, cycles = {"alu": (1024, 10000), "systolic": (8192, 5000)}[wl]
        run = oracle.alu_run if wl == "alu" else oracle.systolic_run
        nchk = min(args.check, lanes)
        ref = np.concatenate([run(seed, nchk, cycles, threads=th),
                              run(seed, nchk, cycles, stim0=lanes - nchk, threads=th)])
        runs = [("fused", cd, MODE_FUSED, args.chunk, 0, 0), ("graph", cd, MODE_GRAPH, args.chunk, 0, 0)]
        if f"{wl}_tuned" in registry.load_index():
            # the autotuner's choice of compile-time options and launch shape
            # (with the multi-wavefront fused kernel when it chose that)
            from rtlflow_amd.autotune import choice
            t = choice(wl)
            runs.append(("tuned", registry.get(f"{wl}_tuned"), MODE_FUSED,
                         t["knobs"].get("chunk", args.chunk), t["knobs"].get("lane_pad", 0),
                         t["knobs"].get("multiwave", 0)))
        if args.main_only:
            runs = runs[-1:]
        for form, c, mode, chunk, pad, mw in runs:
            log(f"[bench] {wl} form={form} lanes={lanes} cycles={cycles} multiwave={mw}")
            with c.model(lanes, fused_chunk=chunk, lane_pad=pad, fused_multiwave=mw) as m:
                m.begin(seed)
                m.run_cycles(0, mode)
                m.sync()
                m.reset_stats()
                t0 = time.perf_counter()
                m.run_cycles(cycles, mode)
                m.sync()
                dt = time.perf_counter() - t0
                st = m.stats()
                h = m.hashes()
            got = np.concatenate([h[:nchk], h[lanes - nchk:]])
            ok = bool((got == ref).all())
            if mode == MODE_FUSED:
                per = st["fused_ms"] / max(1, st["fused_launches"])
                # the committed counters are the reported (last) form's; with
                # a group of 64 stimuli per CU or fewer, a design that has the
                # helped kernel runs it
                hlp = c.manifest.get("help_threads", 0)
                kname = "rf_k_fused_mw" if mw else "rf_k_fused_help" if hlp else "rf_k_fused"
                shape = {"kernel": kname, "lanes": lanes, "cycles_per_launch": min(chunk, cycles),
                         "block": 64 * c.manifest["mw_waves"] if mw else hlp or c.manifest["block"]}
                # stimulus-cycles of the average launch (the last one runs
                # what is left of the workload)
                rl = roofline_line(b_alg, lanes * cycles / max(1, st["fused_launches"]), per, kname,
                                   f"{wl}_{form}_traffic.json", shape, f"{wl}_{form}_sq.json")
            else:
                per = st["graph_ms"] / max(1, st["graph_launches"])
                rl = roofline_line(b_alg, lanes, per, "cycle graph")
            forms[form] = {"seconds": dt, "value": lanes * cycles / dt, "bit_exact_sample": ok,
                           "checked_stimuli": 2 * nchk, "roofline": rl}
            log(f"[bench] form={form} {dt:.3f}s {lanes * cycles / dt:.4g} stim-cycles/s oracle_match={ok}")
        workload = f"{wl}: {lanes} stimuli x {cycles} cycles"
        if args.main_only:
            return print_other(args, wl, man, forms, workload, None)
        ns = args.cpu_sample or lanes       # the whole workload: a second or two on the CPU
        t0 = time.perf_counter()
        run(seed, ns, cycles, threads=th)
        cdt = time.perf_counter() - t0
        cpu = {"value": ns * cycles / cdt, "unit": "stimulus-cycles/s", "cores": th,
               "kind": "port", "nproc": os.cpu_count(),
               "sample": f"{ns} stimuli x {cycles} cycles, C oracle ({cdt:.1f} s)"}
    else:
        nstim, lanes = 16384, args.lanes if args.lanes != 65536 else 8192
        progs = rv32i.programs(seed, np.arange(nstim))
        budgets = rv32i.budgets(seed, nstim)
        total = int(budgets.astype(np.int64).sum())
        nchk = min(args.check, nstim)
        ref = oracle.rv32i_run(progs[:nchk], seed, budgets[:nchk], threads=th)
        libs = [("batched", cd, lanes, 0)]
        if "rv32i_tuned" in registry.load_index():
            # the autotuner's choice: stimuli per block, memory layout, lanes
            # per queue (measured on a quarter-size queue, scaled to this one)
            from rtlflow_amd.autotune import WORKLOADS, choice
            t = choice("rv32i")
            libs.append(("tuned", registry.get("rv32i_tuned"),
                         t["knobs"]["lanes"] * nstim // WORKLOADS["rv32i"]["nstim"],
                         t["knobs"].get("lane_pad", 0)))
        outs = {}
        if args.main_only:
            libs = libs[-1:]
        for form, c, ln, pad in libs:
            log(f"[bench] rv32i {form} queue: {nstim} stimuli on {ln} lanes, {total} stimulus-cycles")
            with c.model(ln, lane_pad=pad) as m:
                m.set_mem_images("imem", progs)
                m.sync()
                m.reset_stats()
                t0 = time.perf_counter()
                out = m.submit_queue(seed, budgets)
                dt = time.perf_counter() - t0
                st = m.stats()
            outs[form] = out
            ok = bool((out[:nchk] == ref).all()) and bool((out == outs.get("batched", out)).all())
            rl = roofline_line(b_alg, total, st["fused_ms"] / max(1, st["fused_launches"]),
                               "rf_k_persistent", f"{wl}_persistent_traffic.json",
                               {"lanes": ln, "stimuli": len(budgets)}, f"{wl}_persistent_sq.json")
            forms[form] = {"seconds": dt, "value": total / dt, "bit_exact_sample": ok,
                           "checked_stimuli": nchk, "lanes": ln, "roofline": rl}
            log(f"[bench] {form} {dt:.3f}s {total / dt:.4g} stim-cycles/s oracle_match={ok}")
        med = int(np.median(budgets))
        gl = 4096
        if args.main_only:
            return print_other(args, wl, man, forms, f"rv32i: {nstim} stimuli, lognormal budgets", None)
        with cd.model(gl) as m:
            m.mem_write("imem", progs[:gl])
            m.begin(seed)
            m.run_cycles(0, MODE_GRAPH)
            m.sync()
            m.reset_stats()
            t0 = time.perf_counter()
            m.run_cycles(med, MODE_GRAPH)
            m.sync()
            dtg = time.perf_counter() - t0
            st = m.stats()
            hg = m.hashes()
        refg = oracle.rv32i_run(progs[:8], seed, [med] * 8, threads=th)
        forms["graph"] = {"seconds": dtg, "value": gl * med / dtg, "bit_exact_sample":
                          bool((hg[:8] == refg).all()), "checked_stimuli": 8, "lanes": gl,
                          "cycles": med,
                          "roofline": roofline_line(b_alg, gl, st["graph_ms"] / max(1, st["graph_launches"]),
                                                    "cycle graph")}
        log(f"[bench] graph {dtg:.3f}s {gl * med / dtg:.4g} stim-cycles/s")
        workload = f"rv32i: {nstim} stimuli, lognormal budgets (median 5000, [1000, 100000]), {total} cycles"
        ns = args.cpu_sample or 4096
        t0 = time.perf_counter()
        oracle.rv32i_run(progs[:ns], seed, budgets[:ns], threads=th)
        cdt = time.perf_counter() - t0
        cpu = {"value": int(budgets[:ns].astype(np.int64).sum()) / cdt, "unit": "stimulus-cycles/s",
               "cores": th, "kind": "port", "nproc": os.cpu_count(),
               "sample": f"{ns} stimuli at their budgets, C oracle ({cdt:.1f} s)"}
    return print_other(args, wl, man, forms, workload, cpu)


def print_other(args, wl, man, forms, workload, cpu):
    exact = {k: v for k, v in forms.items() if v["bit_exact_sample"]}
    # the autotuner's choice is the configured path (its profiles are the
    # committed ones); without one, the fastest bit-exact form
    main_form = "tuned" if "tuned" in exact else max(exact or forms, key=lambda k: forms[k]["value"])
    f = forms[main_form]
    line = {
        "metric": "stimulus-cycles/sec, bit-exact vs Verilator CPU; batched+learned vs plain GPU",
        "value": f["value"], "unit": "stimulus-cycles/s", "n_gpus": 1, "steps": 1,
        "warmup": 0, "ms_per_step": f["seconds"] * 1e3, "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "u32", "data": "synthetic",
        "config": {"workload": workload, "design": wl, "form": main_form, "mtasks": man["mtasks"]},
        "forms": forms, "bit_exact_sample": all(v["bit_exact_sample"] for v in forms.values()),
        "roofline": f["roofline"],
        "cpu_baseline": cpu,
    }
    print(json.dumps(line), flush=True)


def bench_net5s(args):
    """Random netlist with RAMs at one tenth of configuration 5's gate and
    flip-flop counts: 4,096 stimuli with lognormal budgets through the
    batched queue, partitioned by the instruction-count heuristic and by the
    learned cost model, beside the plain per-mtask graph form at the median
    budget."""
    from rtlflow_amd.designs import registry, rv32i
    from rtlflow_amd.model import MODE_BITPLANE, MODE_GRAPH
    import oracle
    seed = registry.SEED_CFG[5]
    nstim = 4096
    lanes = args.lanes if args.lanes != 65536 else nstim
    budgets = rv32i.budgets(seed, nstim, median=2000, lo=200, hi=20000)
    total = int(budgets.astype(np.int64).sum())
    tb = registry.table_bytes("net5s")
    nchk = min(args.check, nstim)
    ref = oracle.netlist_run(tb, seed, nchk, budgets=budgets[:nchk], threads=cpu_threads())
    forms = {}
    hashes = {}
    # the per-lane batched forms take about 7 ms per cycle at this size (one
    # lane per stimulus, 64 wavefronts on the chip): they run the budgets
    # capped at the median, heuristic and learned partitions alike
    capb = np.minimum(budgets, 2000).astype(np.uint32)
    ctotal = int(capb.astype(np.int64).sum())
    cref = oracle.netlist_run(tb, seed, nchk, budgets=capb[:nchk], threads=cpu_threads())
    for form, name in (() if args.main_only else (("batched", "net5s"), ("batched_learned", "net5s_learned"))):
        cd = registry.get(name)
        log(f"[bench] net5s {form}: {nstim} stimuli on {lanes} lanes, budgets capped at 2000 "
            f"({ctotal} stimulus-cycles), {cd.manifest['mtasks']} mtasks")
        with cd.model(lanes) as m:
            m.sync()
            t0 = time.perf_counter()
            out = m.submit_queue(seed, capb)
            dt = time.perf_counter() - t0
        hashes[form] = out
        ok = bool((out[:nchk] == cref).all())
        forms[form] = {"seconds": dt, "value": ctotal / dt, "bit_exact_sample": ok,
                       "checked_stimuli": nchk, "lanes": lanes, "mtasks": cd.manifest["mtasks"],
                       "budgets": "capped at 2000", "stimulus_cycles": ctotal}
        log(f"[bench] {form} {dt:.3f}s {ctotal / dt:.4g} stim-cycles/s oracle_match={ok}")
    if not args.main_only:
        same = bool((hashes["batched"] == hashes["batched_learned"]).all())
        forms["batched_learned"]["same_hashes_as_heuristic"] = same
    cd = registry.get("net5s")
    if cd.manifest.get("bitplane", {}).get("supported"):
        # the bit-plane form: stimuli dealt to 64-lane groups longest budget
        # first, the RAMs as memory ports
        nt = args.bp_threads
        if not nt:
            from rtlflow_amd.autotune import choice
            t = choice("net5s")
            nt = t["knobs"]["bp_threads"] if t and t.get("form") == "bitplane" else 1024
        log(f"[bench] net5s bitplane: {nstim} stimuli on {lanes} lanes, {nt} threads per group")
        with cd.model(lanes, bitplane_threads=nt) as m:
            m.submit_queue(seed, budgets[:64], mode=MODE_BITPLANE)    # code load
            m.sync()
            m.reset_stats()
            t0 = time.perf_counter()
            out = m.submit_queue(seed, budgets, mode=MODE_BITPLANE)
            dt = time.perf_counter() - t0
            st = m.stats()
        ok = bool((out[:nchk] == ref).all())
        # one launch per round of lanes; the useful stimulus-cycles (each
        # stimulus's own budget) over the launches
        b_alg = 2 * ((cd.manifest["bitplane"]["state_bits"] + 7) // 8) + 8 * 16
        rl = roofline_line(b_alg, total / max(1, st["bitplane_launches"]),
                           st["bitplane_ms"] / max(1, st["bitplane_launches"]), f"rf_bp_kernel<{nt}>",
                           "net5s_bitplane_traffic.json", {"lanes": lanes, "bitplane_threads": nt},
                           "net5s_bitplane_sq.json")
        forms["bitplane"] = {"seconds": dt, "value": total / dt, "bit_exact_sample": ok,
                             "checked_stimuli": nchk, "lanes": lanes, "threads": nt,
                             "stimulus_cycles": total, "roofline": rl}
        log(f"[bench] bitplane {dt:.3f}s {total / dt:.4g} stim-cycles/s oracle_match={ok}")
    if args.main_only:
        f = forms["bitplane"]
        print(json.dumps({"metric": "stimulus-cycles/sec, bit-exact vs Verilator CPU; batched+learned vs plain GPU",
                          "value": f["value"], "unit": "stimulus-cycles/s", "n_gpus": 1, "forms": forms,
                          "roofline": f.get("roofline")}), flush=True)
        return
    # the learned partition in the form its cost model predicts (the
    # per-mtask graph form: the sum of an eval's mtask kernel times)
    lc = 200
    lres = {}
    for tag, name in (("heuristic", "net5s"), ("learned", "net5s_learned")):
        c = registry.get(name)
        log(f"[bench] net5s partition={tag} graph form, {nstim} x {lc} cycles, {c.manifest['mtasks']} mtasks")
        with c.model(nstim) as m:
            m.begin(seed)
            m.run_cycles(0, MODE_GRAPH)
            m.sync()
            t0 = time.perf_counter()
            m.run_cycles(lc, MODE_GRAPH)
            m.sync()
            dtl = time.perf_counter() - t0
            lres[tag] = (nstim * lc / dtl, m.hashes(), c.manifest["mtasks"])
    lref = oracle.netlist_run(tb, seed, 8, cycles=lc, threads=8)
    lsame = bool((lres["heuristic"][1] == lres["learned"][1]).all())
    lexact = lsame and bool((lres["learned"][1][:8] == lref).all())
    lsp = lres["learned"][0] / lres["heuristic"][0]
    learned = {"form": "graph", "cycles": lc, "heuristic": lres["heuristic"][0],
               "learned": lres["learned"][0], "heuristic_mtasks": lres["heuristic"][2],
               "learned_mtasks": lres["learned"][2], "speedup": lsp, "bit_exact": lexact,
               "kept": bool(lexact and lsp > 1.0)}
    log(f"[bench] net5s learned/heuristic graph throughput {lsp:.3f} (bit-exact {lexact})")
    med = int(np.median(budgets))
    cd = registry.get("net5s")
    with cd.model(nstim) as m:
        m.begin(seed)
        m.sync()
        t0 = time.perf_counter()
        m.run_cycles(med, MODE_GRAPH)
        m.sync()
        dtg = time.perf_counter() - t0
        hg = m.hashes()
    refg = oracle.netlist_run(tb, seed, 8, cycles=med, threads=8)
    forms["graph"] = {"seconds": dtg, "value": nstim * med / dtg,
                      "bit_exact_sample": bool((hg[:8] == refg).all()), "checked_stimuli": 8,
                      "lanes": nstim, "cycles": med}
    log(f"[bench] graph {dtg:.3f}s {nstim * med / dtg:.4g} stim-cycles/s")
    ns = args.cpu_sample or 128
    t0 = time.perf_counter()
    oracle.netlist_run(tb, seed, ns, budgets=budgets[:ns], threads=cpu_threads())
    cdt = time.perf_counter() - t0
    cpu = {"value": int(budgets[:ns].astype(np.int64).sum()) / cdt, "unit": "stimulus-cycles/s",
           "cores": cpu_threads(), "kind": "port", "nproc": os.cpu_count(),
           "sample": f"{ns} stimuli at their budgets, C oracle"}
    exact = {k: v for k, v in forms.items() if v["bit_exact_sample"]}
    # the autotuner's choice is the configured path (its profiles are the
    # committed ones); without one, the fastest bit-exact form
    main_form = "tuned" if "tuned" in exact else max(exact or forms, key=lambda k: forms[k]["value"])
    f = forms[main_form]
    line = {
        "metric": "stimulus-cycles/sec, bit-exact vs Verilator CPU; batched+learned vs plain GPU",
        "value": f["value"], "unit": "stimulus-cycles/s", "n_gpus": 1, "steps": 1,
        "warmup": args.warmup, "ms_per_step": f["seconds"] * 1e3, "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "integer", "data": "synthetic",
        "config": {"workload": f"net5s: random netlist 50k gates / 5k flops / 8 x 1,024 x 64-bit RAMs / "
                               f"128 PI / 64 PO, {nstim} stimuli, lognormal budgets (median 2000, "
                               f"[200, 20000]), {total} cycles",
                   "design": "net5s", "form": main_form},
        "forms": forms, "bit_exact_sample": all(v["bit_exact_sample"] for v in forms.values()),
        "learned_vs_heuristic": forms["batched_learned"]["value"] / forms["batched"]["value"],
        "judge": {"graph": learned, "batched": {"kept": forms["batched_learned"]["value"] > forms["batched"]["value"]}},
        "learned_partition": learned,
        "roofline": f.get("roofline"),
        "cpu_baseline": cpu,
    }
    print(json.dumps(line), flush=True)


def bench_net5(args):
    """Configuration 5 at its stated size through the gate-net engine: a
    random netlist of 500,000 gates, 50,000 flip-flops, eight 1,024 x 64-bit
    synchronous RAMs, 128 inputs and 64 outputs; 4,096 stimuli with
    lognormal budgets (median 2,000, clipped to [200, 20,000]). The
    bit-plane form runs the whole workload (a step); the plain per-mtask
    graph form runs the heuristic and the learned partitions on a bounded
    number of cycles, and the heuristic judges the learned one."""
    from rtlflow_amd import judge
    from rtlflow_amd.designs import registry, rv32i
    from rtlflow_amd.gatenet import GateNet
    import oracle
    seed = registry.SEED_CFG[5]
    nstim = 4096
    budgets = rv32i.budgets(seed, nstim, median=2000, lo=200, hi=20000)
    if args.budget_cap:
        budgets = np.minimum(budgets, args.budget_cap)
    total = int(budgets.astype(np.int64).sum())
    tb = registry.gatenet_table("net5")
    meta = registry.gatenet_meta("net5")
    th = cpu_threads()
    forms = {}
    log(f"[bench] net5 bitplane: {nstim} stimuli, {total} stimulus-cycles, max budget {int(budgets.max())}")
    with GateNet(registry.gatenet_program("net5"), nstim) as g:
        g.run(GateNet.BITPLANE, seed, np.minimum(budgets, 2))     # level graphs, code load
        t0 = time.perf_counter()
        h, ms = g.run(GateNet.BITPLANE, seed, budgets)
        dt = time.perf_counter() - t0
        nodes = g.nodes_per_cycle(GateNet.BITPLANE)
    nchk = min(args.check, 16)
    ref = np.concatenate([oracle.netlist_run(tb, seed, nchk, budgets=budgets[:nchk], threads=th),
                          oracle.netlist_run(tb, seed, nchk, stim0=nstim - nchk,
                                             budgets=budgets[nstim - nchk:], threads=th)])
    ok = bool((np.concatenate([h[:nchk], h[nstim - nchk:]]) == ref).all())
    # algorithmic bytes: every flip-flop bit read and written once per
    # stimulus-cycle, the RAM words read and written (8 x 2 x 8 B), the
    # inputs and outputs (16 B + 8 B)
    b_alg = 2 * ((50000 + 7) // 8) + 8 * 16 + 24
    # no graph nodes: the run was one launch of the LDS kernel per 16,384 cycles
    # (planned at its start: "seconds" holds the planning, kernel_ms does not)
    launches = -(-(int(budgets.max()) + 1) // 16384)
    rl = roofline_line(b_alg, total / launches, ms / launches, "rf_gnl_kernel", "net5_gatenet_traffic.json",
                       {"lanes": nstim, "longest_budget": int(budgets.max())}, "net5_gatenet_sq.json") if nodes == 0 \
        else roofline_line(b_alg, total, ms, "gate-net bit-plane cycle graph")
    forms["bitplane"] = {"seconds": dt, "value": total / dt, "bit_exact_sample": ok, "checked_stimuli": 2 * nchk,
                         "kernel_ms": ms, "launch": "cycle graph" if nodes else "one kernel per 16,384 cycles",
                         "graph_nodes_per_cycle": nodes, "roofline": rl}
    log(f"[bench] net5 bitplane {dt:.3f}s {total / dt:.4g} stim-cycles/s oracle_match={ok}")
    if args.main_only:
        print(json.dumps({"metric": "stimulus-cycles/sec, bit-exact vs Verilator CPU; batched+learned vs plain GPU",
                          "value": forms["bitplane"]["value"], "unit": "stimulus-cycles/s", "n_gpus": 1,
                          "forms": forms, "roofline": rl}), flush=True)
        return
    # the plain per-mtask graph form: heuristic and learned partitions on
    # the first cycles of the same stimuli
    gc = 8
    gb = np.minimum(budgets, gc)
    gref = oracle.netlist_run(tb, seed, nchk, budgets=gb[:nchk], threads=th)
    res = {}
    for tag in ("heuristic", "learned"):
        if tag not in meta["schedules"]:
            continue
        with GateNet(registry.gatenet_program("net5", tag), nstim) as g:
            g.run(GateNet.GRAPH, seed, np.minimum(budgets, 1))
            t0 = time.perf_counter()
            hg, gms = g.run(GateNet.GRAPH, seed, gb)
            gdt = time.perf_counter() - t0
            mt = g.mtasks()
        res[tag] = (int(gb.astype(np.int64).sum()) / gdt, hg, mt)
        forms[f"graph_{tag}"] = {"seconds": gdt, "value": res[tag][0],
                                 "bit_exact_sample": bool((hg[:nchk] == gref).all()), "checked_stimuli": nchk,
                                 "cycles": gc, "mtasks": mt, "threads": meta["schedules"][tag]["threads"]}
        log(f"[bench] net5 graph {tag} ({mt} mtasks) {gdt:.3f}s {res[tag][0]:.4g} stim-cycles/s")
    learned = None
    if "learned" in res:
        learned = judge.decide(res["heuristic"][0], res["learned"][0], res["heuristic"][1], res["learned"][1],
                               gref, np.arange(nchk))
        learned.update(form="graph", cycles=gc, heuristic_mtasks=res["heuristic"][2],
                       learned_mtasks=res["learned"][2])
    ns = args.cpu_sample or th
    cap = 600
    t0 = time.perf_counter()
    oracle.netlist_run(tb, seed, ns, budgets=np.minimum(budgets[:ns], cap), threads=th)
    cdt = time.perf_counter() - t0
    csc = int(np.minimum(budgets[:ns], cap).astype(np.int64).sum())
    cpu = {"value": csc / cdt, "unit": "stimulus-cycles/s", "cores": min(th, ns), "kind": "port",
           "nproc": os.cpu_count(),
           "sample": f"{ns} stimuli, budgets capped at {cap} ({csc} stimulus-cycles, {cdt:.1f} s), C oracle"}
    f = forms["bitplane"]
    line = {
        "metric": "stimulus-cycles/sec, bit-exact vs Verilator CPU; batched+learned vs plain GPU",
        "value": f["value"], "unit": "stimulus-cycles/s", "n_gpus": 1, "steps": 1, "warmup": 1,
        "ms_per_step": f["seconds"] * 1e3, "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "u64", "data": "synthetic",
        "config": {"workload": f"net5: random netlist 500k gates / 50k flops / 8 x 1,024 x 64-bit RAMs / "
                               f"128 PI / 64 PO, {nstim} stimuli, lognormal budgets (median 2000, "
                               f"[200, 20000]), {total} cycles", "design": "net5", "form": "bitplane"},
        "forms": forms, "bit_exact_sample": all(v["bit_exact_sample"] for v in forms.values()),
        "learned_partition": learned, "roofline": f["roofline"], "cpu_baseline": cpu,
    }
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
