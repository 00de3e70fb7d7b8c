"""Fused kernel with helper wavefronts (rf_k_fused_help).

A workgroup serves 64 stimuli: wavefront 0 runs the design, the wavefronts
behind it draw the input words and fold the output hash, the cycle's other
work. Input words depend on nothing the design computes and the hash feeds
nothing back, so they run a stage of STAGE cycles ahead and behind, through
double-buffered rings in LDS with one barrier a stage.

Measured on the register-file ALU, 4,000 cycles: at 1 to 16,384 stimuli 2.5 to
2.9 ms with one wavefront per 64 stimuli, 2.1 with helpers beside the same
logic, 1.1 with the logic's edge tests and case branches taken out, 0.78 to 0.81
with the launch's first cycle apart and four cycles unrolled; at 32,768 2.9 ->
1.07, at 65,536 3.0 -> 1.68. What is left is the design's dependent chain of
some 70 instructions and two LDS reads a cycle.

For designs whose cycle is mostly that work: a SplitMix64 word is two 64-bit
products (some 45 instructions, the quarter-rate multiplies weighed by four),
a byte of the FNV-1a hash a third of one. In the register-file ALU, five input
words and four hash bytes take about three quarters of a cycle's issue slots
of its one wavefront, while the other SIMDs of the chip are idle.
"""
from __future__ import annotations

import re
from typing import List, Optional, Tuple

from .ir import CLASS_BYTES
from .layout import class_of

# cycles between barriers: the ALU's rings are then 24 KB of LDS, so that four
# groups fit a CU
STAGE = 8
HELPERS = 3        # wavefronts beside the design's: one on each SIMD of a CU
WORD_OPS = 45      # issue slots of an input word, of a hash byte
BYTE_OPS = 15
LDS_MAX = 48 * 1024
CTY = {"C": "uint8_t", "S": "uint16_t", "I": "uint32_t", "Q": "uint64_t"}


def helped_ops(comp) -> int:
    """Issue slots of one cycle's input words and output hash."""
    words = bytes_ = 0
    for p in comp.port_table():
        if p["dir"] == 0:
            words += (p["width"] + 63) // 64
        if p["hashed"]:
            v = p["var"]
            bytes_ += 4 * v.words if v.width > 64 else CLASS_BYTES[class_of(v)]
    return words * WORD_OPS + bytes_ * BYTE_OPS


def emit_fused_help(comp) -> Tuple[Optional[str], int]:
    """(source of rf_k_fused_help, its threads), or (None, 0): the host
    build, the calls form, change-detected variables, wide ports, memories
    outside LDS, state beyond the registers, and designs whose own logic is
    more than twice the helpers' work (the cycle would gain less than a
    third)."""
    from . import compiler as c
    none = (None, 0)
    if comp.host or comp.calls or comp.sch.change_vars:
        return none
    words = c._input_words(comp)
    ports = [p for p in comp.port_table() if p["dir"] == 0]
    outs = [p["var"] for p in comp.port_table() if p["hashed"]]
    if not words or any(p["width"] > 64 for p in ports) or any(v.width > 64 for v in outs):
        return none
    if 2 * helped_ops(comp) < 2 * sum(comp.vcost):
        return none
    d = comp.design
    gen = c.Gen(comp)
    gen.lds = c.lds_memories(comp)
    gen.select_cases = True
    if any(m.is_mem and comp.layout.has(m) and m not in gen.lds for m in d.vars):
        return none
    gen.top_lines = []
    gen.local = c._fused_locals(comp)
    cone = c.clk0_cone(comp)
    c.plan_packing(comp, gen, comp.stored | c.clk0_carried(comp, cone))
    if c.place_lds_state(comp, gen):
        return none
    wide = ["uint64_t" if p["width"] > 32 else "uint32_t" for p in ports]
    lds = sum(m.depth * m.words * CLASS_BYTES[class_of(m)] for m in gen.lds) * 64
    lds += 2 * STAGE * 64 * (sum(8 if t == "uint64_t" else 4 for t in wide) +
                             sum(CLASS_BYTES[class_of(v)] for v in outs))
    if lds > LDS_MAX:
        return none
    for v in sorted(gen.local, key=lambda x: x.id):
        if v in comp.persistent:
            gen.ensure(v)
        else:
            gen.declare(v)
            gen.avail.add(v)
    head, gen.lines = gen.lines, []

    # wavefront 0: a launch's first cycle, and the others: from the second on
    # the last clock values are known (0 after the clk = 0 eval), so the two
    # evals are straight code with no test of an edge left per lane
    def cycle_lines(first: str, unroll: str) -> List[str]:
        for _, n in words:
            gen.emit(f"const uint64_t rfin{n} = ri{n}[b][k][t64];")
        c._stim_code(comp, gen, "0", "0", True, False)
        gen.emit(unroll)
        gen.emit("for (uint32_t ph = 0u; ph < 2u; ++ph) {")
        gen.ind += 1
        for clk in comp.in_clocks:
            gen.emit(gen.set(clk, "ph"))
            gen.dirty.add(clk)
        c._eval_loop_body_split(comp, gen, first, cone)
        gen.ind -= 1
        gen.emit("}")
        for i, v in enumerate(outs):
            gen.ensure(v)
            gen.emit(f"ro{i}[b][k][t64] = ({CTY[class_of(v)]}){gen.get(v)};")
        out, gen.lines = gen.lines, []
        return out

    gen.ind += 4
    cycle0 = cycle_lines("true", "#pragma unroll 1")
    cycle = cycle_lines("false", "#pragma unroll")
    gen.ind -= 4
    # lanes that are done or past the end compute and store nothing: a cycle
    # may touch registers and this lane's LDS columns only
    if any(re.search(r"\bs[CSIQ]\b|\bmb\d|\ba\.|\batomic|\basm\b", ln) for ln in cycle0 + cycle):
        return none
    gen.ind += 1
    c._opaque_bases(gen)
    for v in sorted(gen.dirty | (gen.local & comp.stored), key=lambda x: x.id):
        if v in comp.stored:
            gen.store(v)
    gen.ind -= 1
    tail = gen.lines

    # the helpers' shares: the largest piece to the wavefront with least work
    share: List[Tuple[int, List[int]]] = []
    hash_ops = sum(CLASS_BYTES[class_of(v)] for v in outs) * BYTE_OPS
    H = min(HELPERS, len(words) + 1)
    load = [0] * H
    share = [[] for _ in range(H)]
    load[H - 1] = hash_ops
    for _, n in words:
        w = min(range(H), key=lambda x: load[x])
        load[w] += WORD_OPS
        share[w].append(n)
    keys = {n: key for key, n in words}

    T = 64 * (1 + H)
    L = [f'extern "C" __global__ void __launch_bounds__({T}) rf_k_fused_help(rf_args a) {{']
    L += [ln.replace(f"[{comp.opts.block}];", "[64];") for ln in c._lds_decl_lines(comp, gen.lds)]
    L += [f"    __shared__ {t} ri{n}[2][{STAGE}][64];" for (_, n), t in zip(words, wide)]
    L += [f"    __shared__ {CTY[class_of(v)]} ro{i}[2][{STAGE}][64];" for i, v in enumerate(outs)]
    L += ["    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));",
          "    const uint32_t t64 = threadIdx.x & 63u;",
          "    const uint32_t own = blockIdx.x * 64u + t64;",
          "    const bool live = own < a.nlanes && a.done[own] == 0u;",
          "    if (!__syncthreads_or(live)) return;",
          "    // past the end: the last lane's values, never stored",
          "    const uint32_t lane = own < a.nlanes ? own : a.nlanes - 1u;"]
    pro: List[str] = []
    c._prologue(comp, gen, pro, check_done=False)
    L += pro[2:]
    cp = c._lds_copy_lines(comp, gen.lds, to_lds=True)
    if cp:
        L += ["    if (wave == 0u) {"] + ["    " + ln for ln in cp] + ["    }"]
    L += list(dict.fromkeys(gen.top_lines)) + head
    L += ["    uint64_t h = a.hash[lane];",
          "    const uint32_t cyc = a.cyc[lane];",
          "    const uint64_t sid = (uint64_t)a.stim[lane];",
          f"    const uint32_t stages = (a.ncycles + {STAGE - 1}u) / {STAGE}u;",
          "    // stage s: inputs of s, logic of s - 1, hash of s - 2",
          "    for (uint32_t s = 0u; s < stages + 2u; ++s) {",
          "        if (wave == 0u) {",
          "            if (s >= 1u && s <= stages) {",
          f"                const uint32_t c0 = (s - 1u) * {STAGE}u, b = (s - 1u) & 1u;",
          f"                const uint32_t m = min({STAGE}u, a.ncycles - c0);",
          "                uint32_t k = 0u;",
          "                if (s == 1u) {"]
    L += cycle0
    L += ["                    k = 1u;",
          "                }",
          "                #pragma unroll 4",
          "                for (; k < m; ++k) {"]
    L += cycle
    L += ["                }", "            }", "        }"]
    for w in range(H):
        L.append(f"        if (wave == {w + 1}u) {{")
        if share[w]:
            L += ["            if (s < stages) {",
                  f"                for (uint32_t k = 0u; k < {STAGE}u; ++k) {{",
                  f"                    const uint64_t cy = (uint64_t)(cyc + s * {STAGE}u + k);"]
            L += [f"                    ri{n}[s & 1u][k][t64] = ({wide[n]})rf_stim(a.seed, sid, cy, {keys[n]}u);"
                  for n in share[w]]
            L += ["                }", "            }"]
        if w == H - 1:
            L += ["            if (s >= 2u) {",
                  f"                const uint32_t c0 = (s - 2u) * {STAGE}u, m = min({STAGE}u, a.ncycles - c0);",
                  "                for (uint32_t k = 0u; k < m; ++k) {"]
            L += [f"                    h = rf_fnv_bytes(h, (uint64_t)ro{i}[s & 1u][k][t64], "
                  f"{CLASS_BYTES[class_of(v)]});" for i, v in enumerate(outs)]
            L += ["                }", "            }"]
        L.append("        }")
    L += ["        __syncthreads();", "    }",
          f"    if (wave == {H}u && live) {{",
          "        a.hash[lane] = h;",
          "        a.cyc[lane] = cyc + a.ncycles;",
          "    }",
          "    if (wave == 0u && live) {"]
    L += tail
    L += ["    " + ln for ln in c._lds_copy_lines(comp, gen.lds, to_lds=False)]
    L += ["    }", "}"]
    return "\n".join(L), T
