"""Which of the optional kernels the compiler writes for a design: the helped
fused kernel, packed mtask kernels, the straight batched kernel, the bit-plane
plans. Each falls back to the general kernel without a word, so the GPU tests of
these kernels rest on the designs named here taking them."""
import subprocess
from pathlib import Path

import pytest

import abi_offsets
from rtlflow_amd.compiler import Compiled, Options, emit_source
from rtlflow_amd.designs import registry
from rtlflow_amd.verilog import elaborate

ROOT = Path(__file__).resolve().parent.parent

# design: (threads of the helped kernel, packed mtasks, straight batched kernel)
FORMS = {
    "alu": (256, 0, True),
    "gated": (256, 1, True),
    "kat_shift": (192, 0, False),       # too many wide helpers unrolled: the plain batched kernel
    "kat_signed": (192, 0, True),
    "kat_div": (0, 0, True),
    "mix": (0, 1, True),
    "rams": (0, 0, True),
    "fuzz1": (0, 0, True),
    "fuzz2": (0, 0, True),
    "fuzz3": (0, 0, True),
    "fuzz4": (0, 0, True),
    "net_tiny": (0, -1, True),          # -1: every mtask
    "net_ram": (0, 19, False),          # the other mtasks hold its RAM ports; too long for the straight form
}


@pytest.mark.parametrize("name", FORMS)
def test_forms_of_the_tests_designs(name):
    e = registry.ENTRIES[name]
    spec = e.make()
    comp = Compiled(elaborate(spec["verilog"], spec["top"]), Options(**e.opts))
    text = emit_source(comp)
    man = comp.manifest()
    help_threads, packed, straight = FORMS[name]
    assert man["help_threads"] == help_threads
    assert man["packed_mtasks"] == (man["mtasks"] if packed < 0 else packed)
    assert man["straight_batched"] is straight
    assert ("rf_k_fused_help(rf_args a)" in text) == (help_threads > 0)
    # (the straight form: a stimulus's first cycle in a loop of its own)
    assert ("cyc < min(budget, 1u)" in text) == straight


def test_design_struct_offsets(tmp_path):
    """Where the fields of design ABI 9 and 10 begin (abi_offsets.py)."""
    src = tmp_path / "o.cpp"
    src.write_text('#include <cstddef>\n#include <cstdio>\n#include "rf_design.h"\n'
                   'int main() { printf("%zu %zu %zu %u", offsetof(rf_design, help_threads), '
                   'offsetof(rf_design, bp_plans), sizeof(rf_design), RF_DESIGN_ABI); }\n')
    exe = tmp_path / "o"
    subprocess.run(["g++", "-I", str(ROOT / "include"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    assert [int(x) for x in out.split()] == [abi_offsets.ABI9, abi_offsets.ABI10, abi_offsets.SIZE, abi_offsets.ABI]
