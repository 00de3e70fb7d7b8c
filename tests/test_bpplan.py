"""The planner of the bit-plane kernel's per-cycle program (csrc/rf_bpplan.h)
on the CPU: from random planes, the planned rounds leave the same state
planes, hashed outputs and port operands as the program's own records, in both
record forms and at every workgroup size that plans; no level reads what it
writes, and classed rows carry no inversions."""
import ctypes as C
import subprocess
from pathlib import Path

import numpy as np
import pytest

from rtlflow_amd import bitplane as bp
from rtlflow_amd.build import build_planner
from rtlflow_amd.compiler import Compiled, Options, emit_source
from rtlflow_amd.designs import rams
from rtlflow_amd.designs.fuzz import verilog as fuzz
from rtlflow_amd.designs.netlist import generate
from rtlflow_amd.verilog import elaborate

ROOT = Path(__file__).resolve().parent


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    so = tmp_path_factory.mktemp("bpplan") / "bpplan.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", str(ROOT.parent / "rtlflow_amd" / "csrc"),
                    str(ROOT / "bpplan_host.cpp"), "-o", str(so)], check=True)
    return C.CDLL(str(so))


def plan_run(host, blob, threads, rng):
    b = np.asarray(blob, np.uint32)
    sec = bp.sections(blob)
    s = np.array([sec[k] for k in ("in", "state", "levM", "gatesM", "commitM", "hashM", "portsM")], np.uint32)
    planes = rng.integers(0, 2**64, int(b[2]), dtype=np.uint64)
    planes[0] = 0
    out = [np.zeros(4 * int(b[2]) + 4096, np.uint64) for _ in range(2)]
    info = np.zeros(4, np.uint32)
    ptr = lambda a: a.ctypes.data_as(C.c_void_p)
    rc = host.bpplan_run(ptr(b), ptr(s), threads, ptr(planes), ptr(out[0]), ptr(out[1]), ptr(info))
    return rc, out, info


def sources():
    yield generate(n_gates=3000, n_ff=300, n_pi=64, n_po=64, depth=14, seed=3, name="a")[0]
    yield generate(n_gates=400, n_ff=40, n_pi=16, n_po=24, depth=10, seed=7, name="b")[0]
    yield generate(n_gates=600, n_ff=50, n_pi=70, n_po=20, depth=8, seed=31, n_rams=3, ram_depth=12, ram_width=9,
                   name="c")[0]
    yield rams.verilog()
    for s in range(1, 7):
        yield fuzz(s, name=f"f{s}", bitlevel=True, depth=2)


@pytest.mark.parametrize("byte_form", [True, False])
def test_plans_equal_the_programs_they_are_made_from(host, byte_form, monkeypatch):
    if not byte_form:
        monkeypatch.setattr(bp, "BYTE_FORM_MAX_SLOTS", 0)
    rng = np.random.default_rng(5)
    planned = 0
    for src in sources():
        try:
            blob = bp.encode(bp.compile_program(Compiled(elaborate(src), Options(threads=2))))
        except bp.Unsupported:
            continue
        for threads in (256, 512, 1024):
            rc, (a, b), info = plan_run(host, blob, threads, rng)
            if rc == 1:
                assert info[3] > 40, info
                continue
            assert rc == 0 and (a == b).all(), (rc, threads)
            assert info[0] <= info[3] and info[2] <= info[1], info
            planned += 1
    assert planned >= 12


def test_programs_of_another_form_keep_their_records(host):
    """A hash reference to a state plane (which the commit may change before
    the hash reads it) is not re-planned: every row is a generic record."""
    src = generate(n_gates=400, n_ff=40, n_pi=16, n_po=24, depth=10, seed=7, name="b")[0]
    blob = list(bp.encode(bp.compile_program(Compiled(elaborate(src), Options(threads=2)))))
    sec = bp.sections(blob)
    blob[sec["hashM"] + 2] = blob[sec["commitM"]]
    rc, (a, b), info = plan_run(host, blob, 256, np.random.default_rng(1))
    assert rc == 0 and (a == b).all() and info[1] == info[2]


def _design(name="b"):
    src = generate(n_gates=400, n_ff=40, n_pi=16, n_po=24, depth=10, seed=7, n_rams=1, ram_depth=8, ram_width=4,
                   name=name)[0]
    return Compiled(elaborate(src), Options(threads=2))


def test_design_libraries_carry_their_plans():
    """Planning belongs to the design's build: the emitted source holds the
    plan of every workgroup size that has one, so no model and no run makes
    it."""
    comp = _design()
    text = emit_source(comp)
    for th in bp.PLAN_THREADS:
        words = bp.plan(comp.bitplane_blob, th)
        assert words and f"static const uint32_t rf_bp_plan_{th}[] = {{\n    {words[0]}u, {th}u, {words[2]}u," in text
        assert f"{{{th}u, {len(words)}ull, rf_bp_plan_{th}}}" in text
    assert f"    rf_bp_plans, {len(bp.PLAN_THREADS)}u\n" in text


@pytest.mark.parametrize("byte_form", [True, False])
def test_plans_are_checked_against_their_program(byte_form, monkeypatch):
    """A plan's words pass the check that the runtime makes; a slot, a class,
    a table or a size out of range does not."""
    if not byte_form:
        monkeypatch.setattr(bp, "BYTE_FORM_MAX_SLOTS", 0)
    blob = _design().bitplane_blob
    lib = C.CDLL(str(build_planner()))
    b = np.asarray(blob, np.uint32)
    sec = bp.sections(blob)
    s = np.array([sec[k] for k in bp._PLAN_SECTIONS], np.uint32)
    ptr = lambda a: a.ctypes.data_as(C.c_void_p)
    check = lambda w, th=256: lib.rf_bpplan_check(ptr(b), ptr(s), th, ptr(w), C.c_uint64(len(w)))
    w = np.array(bp.plan(blob, 256), np.uint32)
    assert check(w)
    assert not check(w, 512) and not check(w[:-1]) and not check(w[:8])
    nr, cls, commit, ncom, hsh, ports = (int(w[k]) for k in (2, 5, 6, 7, 8, 9))
    big = int(b[2]) * (8 if byte_form else 1)      # the first slot past the planes

    def bad(at, value):
        v = w.copy()
        v[at] = value
        return not check(v)

    def row(wave, r):                              # first record of the first wavefront row that runs
        return 12 + 2 * (r * 256 + 64 * wave)

    runs = [(wv, r) for wv in range(4) for r in range(nr)
            if (int(w[cls + 8 * wv + 6 + r // 32]) >> (r % 32)) & 1]
    at = row(*runs[0])
    assert bad(at, (int(w[at]) & 0xffff0000) | big) and bad(at, (int(w[at]) & 0xffff) | big << 16)
    if big < 0x8000:
        assert bad(at + 1, (int(w[at + 1]) & 0xffff0000) | big) and bad(at + 1, big << 16)
    assert bad(2, nr + 1) and bad(2, 0) and bad(2, 49)
    assert bad(3, int(w[3]) & ~(1 << (nr - 1)))
    wv, r = runs[0]
    w2 = w.copy()
    for q in range(3):                             # class 7
        w2[cls + 8 * wv + 2 * q] |= 1 << r
    assert not check(w2)
    assert ncom and bad(commit, int(b[2])) and bad(commit + 1, int(b[2])) and bad(commit + 1, 0x80000000 | int(b[2]))
    assert bad(hsh, int(w[hsh]) ^ 1) and bad(hsh + 2, int(b[2])) and bad(ports + 1, int(w[ports + 1]) + 1)
    assert bad(ports + 6, int(b[2])) and bad(ports + 3, 99)
    for k in (5, 6, 7, 8, 9, 10):
        assert bad(k, int(w[k]) + 1) and bad(k, 0xffffffff)
