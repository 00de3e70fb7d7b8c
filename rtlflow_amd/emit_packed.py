"""Packed mtask kernels of the graph form: four lanes per thread.

An mtask of single-bit logic (gate netlists: AND / OR / XOR / NOT / MUX
assignments, flip-flops, constant bit selects of ports) spends one byte load,
one instruction per gate and one byte store per lane. A thread here takes four
lanes: a variable's four bytes are one 32-bit word, a gate one instruction for
all four, an access of a wavefront 256 bytes instead of 64.

``packed_mtask(comp, k)`` returns the kernel's source, or None when the mtask
holds anything else (the per-lane kernel of compiler.emit_mtask_kernel stays).
Values, stores and their order are the per-lane kernel's, so both leave the
same bytes in the state arrays. The grid is the per-lane kernels' (one block
per ``block`` lanes); the first quarter of a block's threads do its lanes.

Measured against the per-lane kernels, us a cycle of the graph form: the
45-mtask netlist 2,130 -> 930 at 65,536 lanes, 1,187 -> 585 at 300; a 780-gate
netlist 433 -> 347 at 65,536, 361 -> 355 at 65 lanes, 359 -> 344 at 1 lane. No
lane count is slower, so every mtask that fits the form takes it.

The statements run in chunks: the loads a chunk needs go out before the chunk
in front of it is computed and stored, so they overlap it (loads complete in
order after the stores before them).
"""
from __future__ import annotations

from typing import Dict, List, Optional, Set, Tuple

from .ir import Assign, Concat, Cond, Const, Expr, Op, Ref, Sel, Var
from .layout import class_of

# Statements of a chunk, and values kept in registers across its end. The
# graph form of the 45-mtask netlist at 65,536 lanes, us a cycle (two evals),
# 2,130 with a byte per lane: 40 / 120 1,143, 24 / 80 963, 12 / 60 929, 6 / 40
# 999, 100 / 220 1,073, 12 / 200 956; at 300 lanes 1,180 to 586. What is left
# is latency: 256 wavefronts a kernel (two lanes a thread, twice as many, 933;
# one, 1,135), one chunk's loads behind the other's stores. The order of 12 /
# 60 and 40 / 120 is the same at 16,384, 4,096 and 300 lanes.
CHUNK = 12
KEEP = 60
# Longer mtasks keep the per-lane kernel: hipcc's time for one straight kernel
# with two instantiations grows faster than its length (a 50,000-gate design
# with 16 of its 44 mtasks above this, up to 960: 381 s per-lane, 662 s all
# packed), and a finer partition of such a design (its learned one has 253 at
# most) has them packed.
STMTS = 500
CTY = {"C": "uint8_t", "S": "uint16_t", "I": "uint32_t", "Q": "uint64_t"}
ARR = {"C": "sC", "S": "sS", "I": "sI", "Q": "sQ"}


class Unpackable(Exception):
    pass


class _Stmt:
    """One assignment: target, right-hand side, clocked edges (or None)."""
    __slots__ = ("var", "rhs", "edges", "reads", "group")

    def __init__(self, var: Var, rhs: Expr, edges, group: int):
        self.var, self.rhs, self.edges, self.group = var, rhs, edges, group
        self.reads: List[Var] = []


def _check(e: Expr, reads: List[Var], wide: Set[Tuple[Var, int]]):
    """A single-bit expression this form evaluates; collects the single-bit
    variables and the (variable, 32-bit word) port words it reads."""
    if e.width != 1:
        raise Unpackable
    if isinstance(e, Const):
        return
    if isinstance(e, Ref):
        if e.var.is_mem or e.var.width != 1:
            raise Unpackable
        if e.var not in reads:
            reads.append(e.var)
        return
    if isinstance(e, Sel):
        if not isinstance(e.a, Ref) or e.a.var.is_mem or not isinstance(e.lsb, int) or e.lsb >= e.a.var.width:
            raise Unpackable
        if e.a.var.width == 1:
            return _check(e.a, reads, wide)
        wide.add((e.a.var, e.lsb // 32))
        return
    if isinstance(e, Cond):
        for x in (e.c, e.a, e.b):
            _check(x, reads, wide)
        return
    if isinstance(e, Op) and e.op in ("and", "or", "xor", "xnor", "not", "logand", "logor", "lognot", "eq", "ne"):
        for x in e.args:
            _check(x, reads, wide)
        return
    raise Unpackable


class _Gen:
    def __init__(self, comp, k: int):
        self.comp = comp
        self.k = k
        self.out: List[str] = []
        self.decl: Dict[Var, bool] = {}
        self.held: Set[Var] = set()       # locals that hold the variable's value
        self.words: Dict[Tuple[Var, int], str] = {}
        self.stmts: List[_Stmt] = []
        self.edges = None
        wide: Set[Tuple[Var, int]] = set()
        written: Set[Var] = set()
        group = 0
        for vid in comp.mtasks[k].vids:
            vx = comp.sch.vertices[vid]
            group += 1
            for p in vx.procs:
                if p.kind not in ("comb", "seq"):
                    raise Unpackable
                edges = None
                if p.kind == "seq":
                    edges = tuple((kind, clk.id) for kind, clk in p.edges)
                    if len(p.edges) != 1 or p.edges[0][0] != "posedge" or (self.edges not in (None, edges)):
                        raise Unpackable
                    self.edges, self.clk = edges, p.edges[0][1]
                elif group and len(vx.procs) != 1:
                    raise Unpackable
                for s in p.stmts:
                    if not isinstance(s, Assign) or not s.lhs.whole or s.lhs.var.is_mem or \
                            s.nb != (p.kind == "seq"):
                        raise Unpackable
                    st = _Stmt(s.lhs.var, s.rhs, edges, group)
                    if s.lhs.var.width == 1:
                        _check(s.rhs, st.reads, wide)
                    elif isinstance(s.rhs, Concat) and s.lhs.var.width <= 64 and edges is None:
                        for x in s.rhs.parts:
                            _check(x, st.reads, wide)
                    else:
                        raise Unpackable
                    written.add(s.lhs.var)
                    self.stmts.append(st)
        if any(v in written for v, _ in wide) or not self.stmts:
            raise Unpackable
        if any(v in written for v in comp.clklast.values()) or \
                (self.edges and (self.clk in written or comp.clklast[self.clk] in written)):
            raise Unpackable
        # clocked assignments of one vertex read the values from before the
        # edge: they must not read each other's targets
        for g in {st.group for st in self.stmts if st.edges}:
            ts = {st.var for st in self.stmts if st.group == g}
            ws = [st for st in self.stmts if st.group == g]
            if len(ts) != len(ws) or any(v in ts and v is not st.var for st in ws for v in st.reads):
                raise Unpackable
        lay = comp.layout
        for st in self.stmts:
            for v in st.reads + [st.var]:
                if v.width == 1 and lay.has(v) and class_of(v) != "C":
                    raise Unpackable
        self.wide = sorted(wide, key=lambda x: (x[0].id, x[1]))

    # --------------------------------------------------------------- output
    def p(self, v: Var) -> str:
        if v not in self.decl:
            self.decl[v] = True
        return f"p{v.id}"

    def addr(self, v: Var, word: int = 0) -> str:
        return f"{ARR[class_of(v)]} + (size_t){self.comp.layout.loc[v] + word} * NP"

    def load(self, v: Var):
        if not self.comp.layout.has(v):
            raise Unpackable
        x = f"rf_pk_ld({self.addr(v)})"
        if v.kind == "input":
            x += " & RF_PK_ONE"
        self.out.append(f"    {self.p(v)} = {x};")
        self.held.add(v)

    def ex(self, e: Expr) -> str:
        if isinstance(e, Const):
            return "RF_PK_ONE" if e.value & 1 else "0u"
        if isinstance(e, Ref):
            return self.p(e.var)
        if isinstance(e, Sel):
            if e.a.var.width == 1:
                return self.p(e.a.var)
            return f"rf_pk_bit(w{e.a.var.id}_{e.lsb // 32}, {e.lsb % 32}u)"
        if isinstance(e, Cond):
            c, a, b = self.ex(e.c), self.ex(e.a), self.ex(e.b)
            return f"(({c} & {a}) | (~{c} & {b}))"
        a = [self.ex(x) for x in e.args]
        if e.op in ("not", "lognot"):
            return f"({a[0]} ^ RF_PK_ONE)"
        if e.op in ("xnor", "eq"):
            return f"({a[0]} ^ {a[1]} ^ RF_PK_ONE)"
        rel = {"and": "&", "logand": "&", "or": "|", "logor": "|", "xor": "^", "ne": "^"}[e.op]
        return f"({a[0]} {rel} {a[1]})"

    def store(self, st: _Stmt, pending: List[str]):
        if st.var in self.comp.stored:
            pending.append(f"    rf_pk_st<FULL>({self.addr(st.var)}, {self.p(st.var)}, m);")

    def wide_store(self, st: _Stmt, pending: List[str]):
        v = st.var
        bits = [self.ex(x) for x in reversed(st.rhs.parts)]
        n = f"b{v.id}"
        self.out.append(f"    const uint32_t {n}[{len(bits)}] = {{{', '.join(bits)}}};")
        if v in self.comp.stored:
            t = CTY[class_of(v)]
            pending.append(f"    for (uint32_t j = 0; j < 4u; ++j)")
            pending.append(f"        if (FULL || ((m >> (8u * j)) & 1u)) ({self.addr(v)})[j] = "
                           f"rf_pk_gather<{t}>({n}, j);")

    def body(self) -> List[str]:
        chunks = [self.stmts[i:i + CHUNK] for i in range(0, len(self.stmts), CHUNK)]
        # a clocked group stays in one chunk
        fixed: List[List[_Stmt]] = []
        for c in chunks:
            while fixed and c and c[0].edges and fixed[-1][-1].group == c[0].group:
                fixed[-1].append(c.pop(0))
            if c:
                fixed.append(c)
        chunks = fixed
        made: List[Set[Var]] = [{st.var for st in c} for c in chunks]
        uses: List[List[Var]] = []
        for c in chunks:
            u: List[Var] = []
            for st in c:
                for v in st.reads:
                    if v not in u:
                        u.append(v)
            uses.append(u)

        def need(i: int) -> List[Var]:
            """Variables chunk i reads that no register holds and that it (or
            the chunk in front, still to be computed) does not make first."""
            first: Set[Var] = set()
            out: List[Var] = []
            for st in chunks[i]:
                for v in st.reads:
                    if v not in first and v not in self.held and v not in out:
                        out.append(v)
                # a clocked target is made only at the edge
                if not st.edges:
                    first.add(st.var)
            return out

        if self.edges:
            for v in (self.clk, self.comp.clklast[self.clk]):
                self.load(v)
            self.out.append(f"    const uint32_t e = {self.p(self.clk)} & ~{self.p(self.comp.clklast[self.clk])}"
                            " & RF_PK_ONE;")
        for v, w in self.wide:
            h = 0 if class_of(v) != "Q" else w
            self.out.append(f"    uint32_t w{v.id}_{w}[4];")
            self.out.append(f"    rf_pk_words({self.addr(v, w if v.width > 64 else 0)}, {h}u, w{v.id}_{w});")
        for v in need(0):
            self.load(v)
        for i, c in enumerate(chunks):
            if i + 1 < len(chunks):
                # the next chunk's loads, but for what this chunk makes
                for v in need(i + 1):
                    if v not in made[i]:
                        self.load(v)
            pending: List[str] = []
            clocked: List[str] = []
            j = 0
            while j < len(c):
                st = c[j]
                if not st.edges:
                    if st.var.width == 1:
                        self.out.append(f"    {self.p(st.var)} = {self.ex(st.rhs)};")
                        self.held.add(st.var)
                        self.store(st, pending)
                    else:
                        self.wide_store(st, pending)
                    j += 1
                    continue
                # a vertex's clocked assignments: all values, then the targets
                g = [x for x in c[j:] if x.group == st.group]
                j += len(g)
                self.out.append("    if (e) {")
                for x in g:
                    self.out.append(f"        const uint32_t d{x.var.id} = {self.ex(x.rhs)};")
                for x in g:
                    v = x.var
                    # lanes without the edge keep the old value
                    self.out.append(f"        {self.p(v)} = FULL ? d{v.id} : rf_pk_sel(e * 255u, "
                                    f"rf_pk_ld({self.addr(v)}), d{v.id});")
                    if v in self.comp.stored:
                        self.out.append(f"        rf_pk_st<FULL>({self.addr(v)}, {self.p(v)}, m);")
                    else:
                        raise Unpackable
                self.out.append("    }")
                # without the edge the local holds nothing new: reread
                for x in g:
                    self.held.discard(x.var)
            self.out += pending
            # a chunk boundary: keep what the next chunks read, soonest first
            if i + 1 < len(chunks):
                keep: List[Var] = []
                for u in uses[i + 1:]:
                    for v in u:
                        if v in self.held and v not in keep:
                            keep.append(v)
                must = {v for v in self.held if not self.comp.layout.has(v) or
                        (v in set().union(*made[:i + 1]) and v not in self.comp.stored)}
                self.held = set(keep[:KEEP]) | must
                late = [v for v in need(i + 1)]
                for v in late:      # made by this chunk's edge, or dropped
                    self.load(v)
        return self.out


def packed_mtask(comp, k: int) -> Optional[str]:
    # whole wavefronts of a quarter block; a change-detecting pass and a host
    # build keep the per-lane kernel
    B = comp.opts.block
    if comp.host or B % 256 or comp.sch.change_vars:
        return None
    try:
        g = _Gen(comp, k)
        if len(g.stmts) > STMTS:
            return None
        body = g.body()
    except Unpackable:
        return None
    full = " && (e == 0u || e == RF_PK_ONE)" if g.edges else ""
    n = f"rf_pk_mtask_{k}"
    out = ["template <bool FULL>",
           f"static __device__ __forceinline__ void {n}(const rf_args& a, uint32_t lane, uint32_t m) {{",
           "    const size_t NP = a.npad;",
           "    uint8_t* const sC = a.c + lane;", "    uint16_t* const sS = a.s + lane;",
           "    uint32_t* const sI = a.i + lane;", "    uint64_t* const sQ = a.q + lane;",
           "    (void)sC; (void)sS; (void)sI; (void)sQ; (void)m;"]
    out += [f"    uint32_t p{v.id} = 0u;" for v in g.decl]
    out += body + ["}",
                   f'extern "C" __global__ void __launch_bounds__({B}) __attribute__((amdgpu_waves_per_eu(1))) '
                   f"rf_mtask_{k}(rf_args a) {{",
                   f"    if (threadIdx.x >= {B // 4}u) return;",
                   f"    const uint32_t lane = blockIdx.x * {B}u + 4u * threadIdx.x;",
                   "    if (lane >= a.nlanes) return;",
                   "    const uint32_t m = rf_pk_active(a.done, lane, a.nlanes);"]
    if g.edges:
        c, last = g.clk, comp.clklast[g.clk]
        out += [f"    const uint32_t e = rf_pk_ld(a.c + (size_t){comp.layout.loc[c]} * a.npad + lane) & "
                f"~rf_pk_ld(a.c + (size_t){comp.layout.loc[last]} * a.npad + lane) & RF_PK_ONE;"]
    out += [f"    if (__all(m == ~0u{full})) {n}<true>(a, lane, m);",
            f"    else {n}<false>(a, lane, m);", "}"]
    return "\n".join(out)
